// Drives the entry points whose blocks run on the matrix cores through the host-only build
// (fake_hip.cpp, fake_kernels.cpp, fake_blocks.cpp): block forwards and backwards of FP32 and BF16
// at the grid sizes where they change kernels, with batches; FP32 and BF16 plans with recomputed
// stencils inside solves; the pair of SM linears; the level combination and the training loss.
// Buffers are allocated at exactly the sizes the interface states.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "fake_hip.hpp"
#include "mlpcg.h"

extern long g_split_calls, g_split_pool, g_split_dots, g_igrad_passes, g_idle_used, g_bf16_images;

namespace {

int g_fail = 0;
#define EXPECT(cond, ...)                                       \
  do {                                                          \
    if (!(cond)) {                                              \
      std::fprintf(stderr, "FAIL %s:%d: ", __FILE__, __LINE__); \
      std::fprintf(stderr, __VA_ARGS__);                        \
      std::fprintf(stderr, "\n");                               \
      ++g_fail;                                                 \
    }                                                           \
  } while (0)
#define OK(call) EXPECT((call) == 0, "%s -> %s", #call, mlpcg_last_error())

struct Buf {
  void* p = nullptr;
  explicit Buf(size_t bytes) {
    if (hipMalloc(&p, bytes) != hipSuccess) std::abort();
    std::memset(p, 0, bytes);
  }
  Buf(const Buf&) = delete;
  ~Buf() { (void)hipFree(p); }
  operator void*() const { return p; }
  template <typename T>
  T* as() const { return (T*)p; }
};

size_t esz(int dt) { return dt == MLPCG_F64 ? 8 : (dt == MLPCG_F32 ? 4 : 2); }

void blocks(int dtype, int C, int B, int n1, int n2, int n3) {
  const size_t V = (size_t)n1 * n2 * n3, s = esz(dtype);
  Buf img(C * V * s), x(B * V * s), y(B * V * s), g(B * V * s), gx(B * V * s);
  Buf W(27 * 27 * C * 4), b(27 * 4), gW(27 * 27 * C * 4), gb(27 * 4);
  Buf ws(mlpcg_sm_block_workspace_size(C, B, n1, n2, n3, dtype));
  OK(mlpcg_sm_block_inference(img, x, W, b, y, ws, C, B, n1, n2, n3, dtype, nullptr));
  OK(mlpcg_sm_block_forward(img, x, W, b, y, ws, C, B, n1, n2, n3, dtype, nullptr));
  OK(mlpcg_sm_block_backward(g, img, x, W, b, gx, gW, gb, ws, C, B, n1, n2, n3, dtype, nullptr));
  OK(mlpcg_sm_block_trans_forward(img, x, W, b, y, ws, C, B, n1, n2, n3, dtype, nullptr));
  OK(mlpcg_sm_block_trans_backward(g, img, x, W, b, gx, gW, gb, ws, C, B, n1, n2, n3, dtype, nullptr));
  if (dtype != MLPCG_BF16) return;
  Buf i16(C * V * 2), pk(mlpcg_fused_pack_bytes(C));
  OK(mlpcg_fused_pack(W.as<float>(), b.as<float>(), C, pk, nullptr));
  for (int k = 0; k < 4; ++k) {
    const void *im = k & 1 ? i16.p : nullptr, *wp = k & 2 ? pk.p : nullptr;
    OK(mlpcg_sm_block_forward_ex(img, im, wp, x, W, b, y, ws, C, B, n1, n2, n3, dtype, nullptr));
    OK(mlpcg_sm_block_backward_ex(g, img, im, wp, x, W, b, gx, gW, gb, ws, C, B, n1, n2, n3, dtype, nullptr));
  }
}

void linear_pair(int dtype, int C, int n1, int n2, int n3) {
  const size_t V = (size_t)n1 * n2 * n3, a = dtype == MLPCG_F64 ? 8 : 4;
  Buf img(C * V * esz(dtype)), w0(27 * C * a), w1(27 * C * a), b0(a), b1(a), z0(a), z1(a), ybar(27 * C * a);
  Buf ws(mlpcg_sm_linear_workspace_size(C, n1, n2, n3, dtype));
  OK(mlpcg_sm_linear_pair(img, w0, b0, z0, w1, b1, z1, ybar, ws, C, n1, n2, n3, dtype, nullptr));
  EXPECT(mlpcg_sm_linear_pair(img, w0, b0, z0, w1, nullptr, z1, ybar, ws, C, n1, n2, n3, dtype, nullptr) != 0, "null bias");
  EXPECT(mlpcg_sm_linear_pair(img, w0, b0, z0, w1, b1, z1, ybar, ws, 4, n1, n2, n3, dtype, nullptr) != 0, "four channels");
}

// a plan of n levels and a solve with it, of every method
void solve(int dtype, int C, int n, int n1, int n2, int n3, int fused_mode) {
  const size_t V = (size_t)n1 * n2 * n3;
  std::vector<Buf*> own;
  std::vector<void*> W, b;
  auto buf = [&](size_t bytes) {
    own.push_back(new Buf(bytes));
    return own.back()->p;
  };
  for (int i = 0; i < 2 * n + 1; ++i) {
    W.push_back(buf(27 * 27 * C * 4));
    b.push_back(buf(27 * 4));
  }
  for (int i = 0; i < 2 * n; ++i) {
    W.push_back(buf(27 * C * 4));
    b.push_back(buf(4));
  }
  Buf img(C * V * 4), flags(V), rhs(4 * V), x(4 * V), x0(4 * V), z(4 * V);
  for (size_t v = 0; v < V; ++v) flags.as<int8_t>()[v] = (int)(v % n3) > n3 / 2 ? 3 : 2;
  mlpcg_precond* P = nullptr;
  OK(mlpcg_precond_create_ex(&P, MLPCG_MODEL_SMALL_SM, n, C, n1, n2, n3, dtype, 0, 0, 0, fused_mode, 1, img, W.data(),
                             b.data(), nullptr));
  mlpcg_solver* S = nullptr;
  OK(mlpcg_solver_create_flags(&S, flags.as<int8_t>(), n1, n2, n3, nullptr));
  for (int method = 0; method < 3; ++method)
    for (int start = 0; start < 2; ++start) {
      mlpcg_solve_info info;
      OK(mlpcg_solver_solve(S, P, rhs.as<float>(), start ? x0.as<float>() : nullptr, x.as<float>(), method, 6, 1e-12, 1e-12,
                            nullptr, &info, nullptr));
      EXPECT(info.iters == 6, "%d iterations", info.iters);
    }
  OK(mlpcg_precond_update(P, img, W.data(), b.data(), nullptr));
  mlpcg_solver_destroy(S);
  mlpcg_precond_destroy(P);
  for (Buf* p : own) delete p;
}

void training(int dtype, int n1, int n2, int n3) {
  const size_t V = (size_t)n1 * n2 * n3, s = esz(dtype);
  Buf x(V * s), y(V * s), o(V * s), c0(4), c1(4), g0(V * s), g1(V * s), out(16), ws(mlpcg_dot_workspace_size());
  OK(mlpcg_comb(x, y, c0, c1, MLPCG_F32, o, (long)V, dtype, nullptr));
  OK(mlpcg_comb_backward(o, x, y, c0, c1, MLPCG_F32, g0, g1, (long)V, dtype, out, MLPCG_F64, ws, nullptr));
  Buf rhs(4 * V), code(V), r(4 * V), coef(8);
  OK(mlpcg_loss_resid(x, dtype, rhs.as<float>(), code.as<uint8_t>(), r.as<float>(), n1, n2, n3, out.as<double>(), ws, nullptr));
  OK(mlpcg_loss_grad(r.as<float>(), code.as<uint8_t>(), coef.as<double>(), g0, dtype, n1, n2, n3, nullptr));
}

}  // namespace

int main() {
  for (int dtype : {MLPCG_F32, MLPCG_BF16, MLPCG_F16, MLPCG_F64}) {
    if (dtype == MLPCG_F64) continue;  // its weights are FP64: the other harness drives it
    for (int C = 1; C <= 3; ++C) {
      blocks(dtype, C, 1, 16, 32, 31);   // below 2^14 voxels
      blocks(dtype, C, 2, 16, 32, 32);   // at it
      blocks(dtype, C, 7, 23, 29, 33);   // several right-hand sides, in passes of the K area's size
      blocks(dtype, C, 3, 16384, 1, 1);  // thin: most edge sums per cell
    }
    blocks(dtype, 1, 1, 64, 64, 64);  // 2^18: the fused apply's
    blocks(dtype, 3, 2, 64, 64, 64);
    blocks(dtype, 1, 1, 72, 72, 64);
  }
  EXPECT(g_split_calls > 0 && g_igrad_passes > 0 && g_bf16_images > 0, "split %ld igrad %ld bf16 %ld", g_split_calls,
         g_igrad_passes, g_bf16_images);
  for (int dtype : {MLPCG_F64, MLPCG_F32, MLPCG_F16, MLPCG_BF16})
    for (int C = 1; C <= 3; ++C) {
      linear_pair(dtype, C, 4, 6, 8);
      linear_pair(dtype, C, 33, 40, 50);
    }
  solve(MLPCG_F32, 1, 1, 64, 64, 68, 1);  // level 0 above 2^18 voxels
  solve(MLPCG_F32, 2, 2, 68, 64, 64, 2);
  EXPECT(g_split_pool > 0 && g_split_dots > 0, "pool %ld dots %ld", g_split_pool, g_split_dots);
  solve(MLPCG_BF16, 1, 2, 72, 64, 64, 1);
  EXPECT(g_idle_used > 0, "idle tiles unused");
  solve(MLPCG_F32, 3, 1, 66, 70, 62, 1);  // stored stencils (several channels below 2^21)
  for (int dtype : {MLPCG_F32, MLPCG_BF16}) training(dtype, 12, 20, 28);
  EXPECT(fakehip::live_device_allocations() == 0, "%ld device allocations left", fakehip::live_device_allocations());
  if (g_fail) return 1;
  std::printf("ALL BLOCK CHECKS PASSED\n");
  return 0;
}
