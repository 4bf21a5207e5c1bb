"""The host-only sanitizer build of build_and_run.py with the stand-ins of the matrix-core blocks
(fake_blocks.cpp, ahead of fake_kernels.cpp) and the harness that drives them."""
from __future__ import annotations

import os
import re
import subprocess

import build_and_run as base

SOURCES = ["fake_blocks.cpp", "harness_blocks.cpp"]
# launchers that only other launchers call (those have stand-ins), or that call another one
INNER = {"launch_wgrad", "launch_sm_linear_noalloc"}


def _obj(src: str) -> str:
    return os.path.join(base.OUT, src + ".o")


def _launchers(objs) -> set:
    """Names of the launch_* functions that objects define."""
    nm = subprocess.run(["nm", "-C", "--defined-only", *objs], capture_output=True, text=True, check=True).stdout
    return set(re.findall(r" T mlpcg::(launch_\w+)\(", nm))


def build() -> str:
    base.build()
    objs = [base._compile(s) for s in SOURCES]
    lib = [_obj(s) for s in base.LIB_SOURCES]
    missing = _launchers(lib) - _launchers([_obj("fake_blocks.cpp"), _obj("fake_kernels.cpp")]) - INNER
    if missing:
        raise RuntimeError(f"launchers without a stand-in: {sorted(missing)}")
    exe = os.path.join(base.OUT, "host_blocks")
    cmd = [base._hipcc(), "--offload-host-only", "-Xarch_host", "-fsanitize=address", "-Xarch_host", "-fsanitize=undefined",
           "-Wl,--allow-multiple-definition", "-o", exe, *objs, _obj("fake_kernels.cpp"), _obj("fake_hip.cpp"), *lib,
           os.path.join(base.OUT, "fatbin_stubs.o")]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed: {' '.join(cmd)}\n{res.stderr}")
    return exe
