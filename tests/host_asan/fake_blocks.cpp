// Stand-ins, as those of fake_kernels.cpp, for the launchers of the matrix-core blocks (split.hpp,
// igrad.hpp), the idle tiles, the level combination and the training loss; and those of
// fake_kernels.cpp whose kernels take other extents now (linked ahead of it): the solver's star
// kernels with runs of at most four cells and half of the partial rows, and the fused apply with
// BF16 images and idle tiles.
#include <sanitizer/asan_interface.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../mlpcg_amd/csrc/kernels.hpp"
#include "../../mlpcg_amd/csrc/pcg.hpp"
#include "fake_hip.hpp"

namespace {

using namespace mlpcg;

void check_region(const char* who, const void* p, size_t bytes) {
  if (p == nullptr || bytes == 0) return;
  void* bad = __asan_region_is_poisoned(const_cast<void*>(p), bytes);
  if (bad) {
    std::fprintf(stderr, "fake kernel %s: %zu-byte extent at %p reaches a bad byte at %p\n", who, bytes, p, bad);
    volatile char c = *(volatile char*)bad;  // ASan reports this access
    (void)c;
    std::abort();
  }
}
#define RD(p, n) check_region(who, (p), (size_t)(n))
#define WR(p, n) check_region(who, (p), (size_t)(n))

void need(bool ok, const char* who, const char* what) {
  if (ok) return;
  std::fprintf(stderr, "fake kernel %s: %s\n", who, what);
  std::abort();
}

size_t esz(int dt) { return dt == kF64 ? 8 : (dt == kF32 ? 4 : 2); }
bool done_now(const int* done) { return done != nullptr && *done != 0; }
bool aligned(const void* p, size_t n) { return ((uintptr_t)p & (n - 1)) == 0; }

void partials_check(const char* who, const double* partials, int rows, unsigned nb) {
  need((size_t)rows * nb * sizeof(double) <= reduction_workspace_bytes(), who, "partials exceed the reduction workspace");
  WR(partials, (size_t)rows * nb * sizeof(double));
}

// star kernels: a run of at most 4 cells per thread, at most half of the 16384 workgroups
unsigned star_blocks(const FlatArgs& a) {
  const int vz = a.n3 % 4 == 0 ? 4 : (a.n3 % 2 == 0 ? 2 : 1);
  const long nb = ((long)a.n1 * a.n2 * (a.n3 / vz) + 255) / 256;
  return (unsigned)std::max(1L, std::min(nb, 8192L));
}

// residual finalize: the emulated residual halves per iteration
void fin_resid(SolveState* st, int init) {
  const char* who = "finalize";
  WR(st, sizeof(SolveState));
  if (init) {
    st->iter = st->done = 0;
    st->norm_b = st->norm = st->rr = st->scale = 1.0;
  } else {
    st->iter += 1;
    st->norm = std::ldexp(1.0, -st->iter);
    st->rr = st->norm * st->norm;
    st->scale = 1.0 / st->norm;
    const double stop = std::fmax(st->tol, st->atol / st->norm_b);
    const bool cont = (st->method == kNpsd) ? !(st->norm < stop) : (st->norm > stop);
    st->done = (cont && st->iter < st->max_it) ? 0 : 1;
  }
  if (st->history && st->iter <= st->max_it) {
    WR(st->history + st->iter, sizeof(double));
    st->history[st->iter] = st->norm;
  }
}

}  // namespace

// calls of the stand-ins that the harness asks after
long g_split_calls = 0, g_split_pool = 0, g_split_dots = 0, g_igrad_passes = 0, g_idle_used = 0, g_bf16_images = 0;

namespace mlpcg {

int launch_resid_flat(const FlatArgs& a, int init, hipStream_t st) {
  fakehip::enqueue(st, [=] {
    const char* who = "resid_flat";
    if (!init && a.st->done) return;
    const long V = (long)a.n1 * a.n2 * a.n3;
    RD(a.code, V);
    RD(a.b, 4 * V);
    RD(a.x_old, 4 * V);
    if (!init) {
      RD(a.p, 4 * V);
      WR(a.x_new, 4 * V);
    }
    WR(a.r, 4 * V);
    partials_check(who, a.partials, 2, star_blocks(a));
    fin_resid(a.st, init);
  });
  return 0;
}

int launch_p_spmv_flat(const FlatArgs& a, hipStream_t st) {
  fakehip::enqueue(st, [=] {
    const char* who = "p_spmv_flat";
    if (a.st->done) return;
    const long V = (long)a.n1 * a.n2 * a.n3;
    RD(a.code, V);
    RD(a.z, 4 * V);
    RD(a.p_old, 4 * V);
    WR(a.p_new, 4 * V);
    WR(a.w, 4 * V);
    partials_check(who, a.partials, 1, star_blocks(a));
  });
  return 0;
}

int launch_npsd_dir_flat(const FlatArgs& a, const float* pN, double* alfa_out, hipStream_t st) {
  fakehip::enqueue(st, [=] {
    const char* who = "npsd_dir_flat";
    if (a.st->done) return;
    const long V = (long)a.n1 * a.n2 * a.n3;
    RD(a.code, V);
    RD(a.z, 4 * V);
    RD(a.r, 4 * V);
    if (pN) RD(pN, 4 * V);
    if (pN && a.p_old) RD(a.p_old, 4 * V);
    WR(a.p_new, 4 * V);
    WR(a.w, 4 * V);
    partials_check(who, a.partials, 3, star_blocks(a));
    WR(alfa_out, sizeof(double));
    *alfa_out = 1.0;
  });
  return 0;
}

int launch_idle_tiles(const uint8_t* code, uint8_t* idle, int n1, int n2, int n3, hipStream_t st) {
  fakehip::enqueue(st, [=] {
    const char* who = "idle_tiles";
    RD(code, (size_t)n1 * n2 * n3);
    WR(idle, idle_tiles_bytes(n1, n2, n3));
    std::memset(idle, 0, idle_tiles_bytes(n1, n2, n3));
  });
  return 0;
}

int launch_sm_fused(int tw, int tx, int ty, int C, const FusedArgs& a, hipStream_t st) {
  MLPCG_REQUIRE(tw == kBF16 && fused_eligible(C, 1, a.n1, a.n2, a.n3), "sm_fused: not eligible");
  const size_t V = (size_t)a.n1 * a.n2 * a.n3;
  const unsigned nb = fused_blocks(C, a.n1, a.n2, a.n3);
  fakehip::enqueue(st, [=] {
    const char* who = "sm_fused";
    if (done_now(a.done)) return;
    need(!a.img_bf16 || (tx == kBF16 && ty == kBF16 && !a.prev && !a.mask_a && !a.mask_b && !a.partials && !a.pool_out),
         who, "a BF16 image with an epilogue");
    g_bf16_images += a.img_bf16 ? 1 : 0;
    RD(a.img, C * V * 2);
    RD(a.apack, fused_weights_bytes(C));
    RD(a.x, V * esz(tx));
    WR(a.y, V * esz(ty));
    if (a.idle) {
      // a byte per 2 x 8 x 64 cells; a cleared tile needs a zero input or the fluid as its mask
      RD(a.idle, idle_tiles_bytes(a.n1, a.n2, a.n3));
      need(tx == kF32 || a.mask_b, who, "idle tiles of a block whose output stays");
      ++g_idle_used;
    }
    if (a.pool_out) WR(a.pool_out, V / 8 * esz(ty));
    if (a.prev) {
      RD(a.prev, V * 2);
      RD(a.c0, 4);
      RD(a.c1, 4);
    }
    if (a.mask_a) RD(a.mask_a, V);
    if (a.mask_b) RD(a.mask_b, V);
    if (a.in_scale) RD(a.in_scale, 8);
    if (a.dot0) {
      RD(a.dot0, 4 * V);
      if (a.dot1) RD(a.dot1, 4 * V);
      partials_check(who, a.partials, 2, nb);
    }
  });
  return 0;
}

int launch_split_pack(const void* W, const void* b, int C, void* pack, hipStream_t st) {
  MLPCG_REQUIRE(C >= 1 && C <= 3, "split_pack: C");
  fakehip::enqueue(st, [=] {
    const char* who = "split_pack";
    RD(W, 27 * 27 * C * 4);
    RD(b, 27 * 4);
    need(aligned(pack, 16), who, "misaligned packing");
    WR(pack, split_pack_bytes(C));
  });
  return 0;
}

int launch_sm_split(int C, const SplitArgs& a, hipStream_t st) {
  MLPCG_REQUIRE(split_eligible(C, a.n1, a.n2, a.n3), "sm_split: not eligible");
  const size_t V = (size_t)a.n1 * a.n2 * a.n3, s = a.is_bf16 ? 2 : 4;
  const unsigned nb = split_blocks(C, a.n1, a.n2, a.n3);
  fakehip::enqueue(st, [=] {
    const char* who = "sm_split";
    if (done_now(a.done)) return;
    const bool epi = a.prev || a.mask_a || a.mask_b || a.partials;
    need(a.B >= 1 && (!epi || (a.B == 1 && !a.is_bf16)), who, "an epilogue with several right-hand sides or BF16");
    ++g_split_calls;
    RD(a.img, C * V * s);
    need(aligned(a.pack, 16), who, "misaligned packing");
    RD(a.pack, split_pack_bytes(C));
    RD(a.x, a.B * V * s);
    WR(a.y, a.B * V * s);
    if (a.prev) {
      RD(a.prev, 4 * V);
      RD(a.c0, 4);
      RD(a.c1, 4);
    }
    if (a.mask_a) RD(a.mask_a, V);
    if (a.mask_b) RD(a.mask_b, V);
    if (a.in_scale) RD(a.in_scale, 8);
    if (a.partials) {
      RD(a.dot0, 4 * V);
      if (a.dot1) RD(a.dot1, 4 * V);
      partials_check(who, a.partials, 2, nb);
      ++g_split_dots;
    }
    if (a.pool_out) {
      need(!epi && a.n1 % 2 == 0 && a.n2 % 2 == 0 && a.n3 % 2 == 0, who, "a pooled output of an odd grid or with an epilogue");
      WR(a.pool_out, V / 8 * 4);
      ++g_split_pool;
    }
  });
  return 0;
}

int launch_igrad(int dtype, const void* img, const void* pack, const void* g, void* dx, void* work, size_t bytes, int C,
                 int B, int n1, int n2, int n3, hipStream_t st) {
  MLPCG_REQUIRE(split_eligible(C, n1, n2, n3) && (dtype == kF32 || dtype == kBF16), "igrad: not eligible");
  const size_t V = (size_t)n1 * n2 * n3, s = esz(dtype);
  const size_t edge = (size_t)n1 * n2 * ((n3 + 63) / 64) * 8 * sizeof(float);
  fakehip::enqueue(st, [=] {
    const char* who = "igrad";
    const int most = (int)std::min<size_t>(bytes / fused_sgrad_bytes(n1, n2, n3), 65535);
    need(most >= 1, who, "a workspace below one right-hand side's sums");
    RD(img, C * V * s);
    RD(pack, split_pack_bytes(C));
    for (int b = 0; b < B; b += most) {  // T [nb][3][V] and the tiles' edge sums, FP32
      const size_t nb = (size_t)std::min(most, B - b);
      RD((const char*)g + b * V * s, nb * V * s);
      const size_t t = (nb * 3 * V * 4 + 255) & ~(size_t)255;
      need(t + nb * edge <= bytes, who, "sums beyond the workspace");
      WR(work, t + nb * edge);
      WR((char*)dx + b * V * s, nb * V * s);
      ++g_igrad_passes;
    }
  });
  return 0;
}

int launch_comb(int dt, const void* x0, const void* x1, const void* c0, const void* c1, int ct, void* y, long n,
                hipStream_t st) {
  MLPCG_REQUIRE(ct == kF32 || ct == kBF16, "comb: coefficients");
  fakehip::enqueue(st, [=] {
    const char* who = "comb";
    if (n == 0) return;
    RD(x0, n * esz(dt));
    RD(x1, n * esz(dt));
    RD(c0, esz(ct));
    RD(c1, esz(ct));
    WR(y, n * esz(dt));
  });
  return 0;
}

int launch_comb_grad(int dt, const void* g, const void* x0, const void* x1, const void* c0, const void* c1, int ct,
                     void* g0, void* g1, long n, double* partials, void* out2, int out_dt, hipStream_t st) {
  MLPCG_REQUIRE((ct == kF32 || ct == kBF16) && (out_dt == kF64 || out_dt == kF32), "comb_grad: types");
  fakehip::enqueue(st, [=] {
    const char* who = "comb_grad";
    RD(g, n * esz(dt));
    RD(x0, n * esz(dt));
    RD(x1, n * esz(dt));
    RD(c0, esz(ct));
    RD(c1, esz(ct));
    if (g0) WR(g0, n * esz(dt));
    if (g1) WR(g1, n * esz(dt));
    // at most one element per thread and 16384 workgroups
    partials_check(who, partials, 2, (unsigned)std::max(1L, std::min((n + 255) / 256, 16384L)));
    WR(out2, 2 * esz(out_dt));
  });
  return 0;
}

int launch_loss_resid(int tx, const void* x, const float* b, const uint8_t* code, float* r, int n1, int n2, int n3,
                      double* partials, double* out2, hipStream_t st) {
  MLPCG_REQUIRE(tx == kF32 || tx == kBF16, "loss_resid: x");
  const size_t V = (size_t)n1 * n2 * n3;
  fakehip::enqueue(st, [=] {
    const char* who = "loss_resid";
    RD(x, V * esz(tx));
    RD(b, 4 * V);
    RD(code, V);
    WR(r, 4 * V);
    const int vz = n3 % 8 == 0 ? 8 : (n3 % 4 == 0 ? 4 : (n3 % 2 == 0 ? 2 : 1));
    const long nb = ((long)n1 * n2 * (n3 / vz) + 255) / 256;
    partials_check(who, partials, 2, (unsigned)std::max(1L, std::min(nb, 16384L)));
    WR(out2, 16);
  });
  return 0;
}

int launch_loss_grad(int tg, const float* r, const uint8_t* code, const double* coef, void* g, int n1, int n2, int n3,
                     hipStream_t st) {
  const size_t V = (size_t)n1 * n2 * n3;
  fakehip::enqueue(st, [=] {
    const char* who = "loss_grad";
    RD(r, 4 * V);
    RD(code, V);
    RD(coef, 8);
    WR(g, V * esz(tg));
  });
  return 0;
}

}  // namespace mlpcg
