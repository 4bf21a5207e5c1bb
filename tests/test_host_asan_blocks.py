"""Host code of the matrix-core blocks, their plans and solves under the host sanitizers
(tests/host_asan/harness_blocks.cpp); every launcher of the library has a stand-in that checks the
extents its kernels touch.  CPU only."""
import os
import shutil
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

pytestmark = pytest.mark.skipif(not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")),
                                reason="needs hipcc for the host-only build")


def test_blocks_clean_under_host_sanitizers():
    sys.path.insert(0, os.path.join(HERE, "host_asan"))
    import build_and_run
    import build_blocks
    res = build_and_run.run(build_blocks.build())
    assert res.returncode == 0, res.stdout[-3000:] + res.stderr[-6000:]
    assert "ALL BLOCK CHECKS PASSED" in res.stdout
