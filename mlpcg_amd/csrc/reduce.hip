// Reductions of the SM preconditioner: the SMLinear mean patch (forward) and the SM
// block weight gradient (backward).  Both are deterministic two-pass reductions
// (block partials in a workspace, then one ordered pass), with no global atomics.
//
//   mean patch  ybar[s,e] = (1/V) sum_v img[s, v+e]          sm_linear_3d_kernel.cu:62-83
//               z = sum_{s,e} w[s,e] ybar[s,e] + b           sm_linear_3d_kernel.cu:185-186
//   weight grad G_p(v) = sum_b a[b,v] c[b,v+d_p]              sm_block_3d_kernel.cu:121-229
//               gW[p,s,e] = sum_v G_p(v) img[s,v+e], gb[p] = sum_v G_p(v)
//               i.e. the [27 x V] . [V x (27C+1)] product of per-voxel outer products:
//               on the matrix cores (wgrad.hpp; BF16 segments of 64 cells by the kernel here),
//               FP64 tiled through LDS with a 3x4 register tile per thread.
#include <mutex>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace mlpcg {

// ---------------------------------------------------------------------------
// Mean patch.  A voxel u contributes to ybar[s,e] iff u - e is inside the grid, i.e.
// per axis: e = -1 excludes the last cell, e = 0 none, e = +1 the first.  So the 27 sums
// add up from those over the grid's disjoint parts T[a1][a2][a3], a in {middle, first, last}
// per axis: its inside, faces, edges and corners (taken away from a total instead, an infinite
// cell would make NaN of the sums without it, and a large one would cost them their digits).
// An interior row only adds to T[0][0][.]; the rows of the faces take a branch, so the pass
// over the image is bound by its loads (adding every run to 27 masked sums was VALU-bound).
// The only cell of an axis counts as middle.  All sums are FP64.  Each
// sum of a workgroup leaves its wave by DPP adds: 27 C butterflies over __shfl_xor, an LDS
// round trip per step, took 20 us on a grid of any size with C = 3.  Whole call, FP32,
// before -> now: 256^3 C = 1 56 -> 23 us, C = 3 176 -> 48 us; 128^3 C = 3 151 -> 21 us;
// below that the launches and their host side remain (C = 3, 16^3: 34 -> 20 us).
// ---------------------------------------------------------------------------
constexpr int kPatchBlocks = 512;       // workgroups of the partial sums at most (two per CU)
constexpr long kPatchOneRuns = 1 << 12;  // grids of at most this many z-runs take one workgroup

template <int C>
struct PatchSums {
  double t[C][27];
};

// the sum over the wave (valid in lane 63) of values that are often zero in all of it: most waves
// touch no face across i, many none across j
__device__ __forceinline__ double wave_sum_sparse(double v) {
  return __builtin_amdgcn_ballot_w64(v != 0.0) == 0 ? 0.0 : wave_sum_dpp(v);
}

template <typename TI, int C, int VZ>
__device__ __forceinline__ void patch_accumulate(const TI* __restrict__ img, int n1, int n2, int n3, unsigned first,
                                                 unsigned stride, PatchSums<C>& p) {
#pragma unroll
  for (int s = 0; s < C; ++s)
#pragma unroll
    for (int o = 0; o < 27; ++o) p.t[s][o] = 0.0;
  const long V = (long)n1 * n2 * n3;
  const unsigned n3c = (unsigned)(n3 / VZ);
  const long nch = (long)n1 * n2 * n3c;
  typedef typename AccOf<TI>::type A;
  A next[C][VZ];  // loaded a run ahead
  auto load = [&](long cid) {
#pragma unroll
    for (int s = 0; s < C; ++s) load_vec<VZ>(img + s * V + cid * VZ, next[s]);
  };
  if (first < nch) load(first);
  for (long cid = first; cid < nch; cid += stride) {
    A run[C][VZ];
#pragma unroll
    for (int s = 0; s < C; ++s)
#pragma unroll
      for (int u = 0; u < VZ; ++u) run[s][u] = next[s][u];
    load(cid + stride < nch ? cid + stride : nch - 1);
    unsigned i, j, kc;
    if (nch <= 0xffffffffL) {  // uniform; 64-bit divisions take a hundred instructions more
      const unsigned row = (unsigned)cid / n3c;
      kc = (unsigned)cid - row * n3c;
      i = row / (unsigned)n2;
      j = row - i * (unsigned)n2;
    } else {
      const long row = cid / n3c;
      kc = (unsigned)(cid - row * n3c);
      i = (unsigned)(row / n2);
      j = (unsigned)(row - (long)i * n2);
    }
    const bool zf = kc == 0 && n3 > 1, zl = kc == n3c - 1 && n3 > 1;
    const int a1 = n1 == 1 ? 0 : i == 0 ? 1 : (int)i == n1 - 1 ? 2 : 0;
    const int a2 = n2 == 1 ? 0 : j == 0 ? 1 : (int)j == n2 - 1 ? 2 : 0;
#pragma unroll
    for (int s = 0; s < C; ++s) {
      const A(&v)[VZ] = run[s];
      // (of one cell that is first or last, the middle keeps nothing)
      double mid = (double)(zf || (VZ == 1 && zl) ? A(0) : v[0]);
#pragma unroll
      for (int u = 1; u < VZ; ++u) mid += (double)(u == VZ - 1 && zl ? A(0) : v[u]);
      const double t3[3] = {mid, (double)(zf ? v[0] : A(0)), (double)(zl ? v[VZ - 1] : A(0))};
      const int part = 3 * a1 + a2;
      if (part == 0) {
#pragma unroll
        for (int u = 0; u < 3; ++u) p.t[s][u] += t3[u];
      }
      int face = part;  // opaque: as one if and else the two take twice the registers
      asm volatile("" : "+v"(face));
      if (face != 0) {
#pragma unroll
        for (int a = 1; a < 9; ++a)
#pragma unroll
          for (int u = 0; u < 3; ++u) p.t[s][3 * a + u] += face == a ? t3[u] : 0.0;
      }
    }
  }
}

// ybar = (sums over the parts that an offset leaves inside the grid) / V, then z0 = w0 . ybar + b0 and, if
// w1 is given, z1 = w1 . ybar + b1: c0 and c1 of one level share their mean patch
// (sm_model_3d.py:236-239 evaluates both on the same image), so one reduction serves both.
// Run by threads 0 .. 127 of the workgroup that holds T in LDS; red: 4 doubles of LDS.
template <typename A>
__device__ __forceinline__ void patch_finish(const double* T, double* red, int n1, int n2, int n3, int NV, double invV,
                                             const A* __restrict__ w0, const A* __restrict__ b0, A* __restrict__ z0,
                                             const A* __restrict__ w1, const A* __restrict__ b1, A* __restrict__ z1,
                                             A* __restrict__ ybar) {
  const int o = threadIdx.x;
  double c0 = 0.0, c1 = 0.0;
  if (o < NV) {
    const double* t = T + (o / 27) * 27;
    const int e = o % 27;
    // whether part a of an axis of n cells counts for offset d - 1
    auto has = [](int d, int a, int n) { return d == 1 || (n > 1 && a != (d == 0 ? 2 : 1)); };
    double s = 0.0;
#pragma unroll
    for (int a = 0; a < 27; ++a) {
      const double v = t[a];
      if (has(e / 9, a / 9, n1) && has(e / 3 % 3, a / 3 % 3, n2) && has(e % 3, a % 3, n3)) s += v;
    }
    const A yb = (A)(s * invV);
    ybar[o] = yb;
    c0 = (double)w0[o] * (double)yb;
    if (w1) c1 = (double)w1[o] * (double)yb;
  }
  c0 = wave_sum_dpp(c0);
  c1 = wave_sum_dpp(c1);
  if (o < 128 && (o & 63) == 63) {
    red[2 * (o >> 6)] = c0;
    red[2 * (o >> 6) + 1] = c1;
  }
  __syncthreads();
  if (o == 0) {
    z0[0] = (A)(red[0] + red[2] + (double)b0[0]);
    if (w1) z1[0] = (A)(red[1] + red[3] + (double)b1[0]);
  }
}

// Workgroup sums of the grid's runs; partials [27 C][gridDim.x].
template <typename TI, int C, int VZ>
__global__ __launch_bounds__(kThreads) void mean_patch_partial_kernel(const TI* __restrict__ img, int n1, int n2,
                                                                      int n3, double* __restrict__ partials) {
  PatchSums<C> p;
  patch_accumulate<TI, C, VZ>(img, n1, n2, n3, blockIdx.x * kThreads + threadIdx.x, gridDim.x * kThreads, p);
  __shared__ double sh[27 * C][4];
  const int w = threadIdx.x >> 6;
#pragma unroll
  for (int o = 0; o < 27 * C; ++o) {
    const double s = wave_sum_sparse(p.t[o / 27][o % 27]);
    if ((threadIdx.x & 63) == 63) sh[o][w] = s;
  }
  __syncthreads();
  for (int o = threadIdx.x; o < 27 * C; o += kThreads)
    partials[(size_t)o * gridDim.x + blockIdx.x] = (sh[o][0] + sh[o][1]) + (sh[o][2] + sh[o][3]);
}

// One wave per sum (coalesced over the workgroups' partials, the loads of a sum in flight
// together), then the patch and its products.
constexpr int kPatchFinalThreads = 1024;
template <typename A>
__global__ __launch_bounds__(kPatchFinalThreads) void mean_patch_final_kernel(
    const double* __restrict__ partials, int nblk, int n1, int n2, int n3, int NV, double invV, const A* __restrict__ w0,
    const A* __restrict__ b0, A* __restrict__ z0, const A* __restrict__ w1, const A* __restrict__ b1,
    A* __restrict__ z1, A* __restrict__ ybar) {
  __shared__ double T[27 * 3], red[4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int o = wv; o < NV; o += kPatchFinalThreads / 64) {
    double a[kPatchBlocks / 64];
#pragma unroll
    for (int u = 0; u < kPatchBlocks / 64; ++u)  // (a uniform test: the loads are in flight together)
      a[u] = 64 * u < nblk ? partials[(size_t)o * nblk + min(lane + 64 * u, nblk - 1)] : 0.0;
#pragma unroll
    for (int u = 0; u < kPatchBlocks / 64; ++u) a[u] = lane + 64 * u < nblk ? a[u] : 0.0;
#pragma unroll
    for (int u = 1; u < kPatchBlocks / 64; ++u) a[0] += a[u];
    const double s = wave_sum_dpp(a[0]);
    if (lane == 63) T[o] = s;
  }
  __syncthreads();
  patch_finish<A>(T, red, n1, n2, n3, NV, invV, w0, b0, z0, w1, b1, z1, ybar);
}

// Small grids: sums, patch and products in one workgroup (one launch instead of two).
template <typename TI, int C, int VZ>
__global__ __launch_bounds__(kPatchFinalThreads) void mean_patch_one_kernel(
    const TI* __restrict__ img, int n1, int n2, int n3, double invV, const typename AccOf<TI>::type* __restrict__ w0,
    const typename AccOf<TI>::type* __restrict__ b0, typename AccOf<TI>::type* __restrict__ z0,
    const typename AccOf<TI>::type* __restrict__ w1, const typename AccOf<TI>::type* __restrict__ b1,
    typename AccOf<TI>::type* __restrict__ z1, typename AccOf<TI>::type* __restrict__ ybar) {
  typedef typename AccOf<TI>::type A;
  constexpr int NW = kPatchFinalThreads / 64;
  __shared__ double sh[27 * C][NW], T[27 * C], red[4];
  const int w = threadIdx.x >> 6;
#pragma unroll 1
  for (int s = 0; s < C; ++s) {  // a channel at a time: 1024 threads leave 128 registers each
    PatchSums<1> p;
    patch_accumulate<TI, 1, VZ>(img + (long)s * n1 * n2 * n3, n1, n2, n3, threadIdx.x, kPatchFinalThreads, p);
#pragma unroll
    for (int o = 0; o < 27; ++o) {
      const double v = wave_sum_sparse(p.t[0][o]);
      if ((threadIdx.x & 63) == 63) sh[27 * s + o][w] = v;
    }
  }
  __syncthreads();
  for (int o = threadIdx.x; o < 27 * C; o += kPatchFinalThreads) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < NW; ++k) s += sh[o][k];
    T[o] = s;
  }
  __syncthreads();
  patch_finish<A>(T, red, n1, n2, n3, 27 * C, invV, w0, b0, z0, w1, b1, z1, ybar);
}

static int mean_patch_vz(int n3) { return (n3 % 4 == 0) ? 4 : (n3 % 2 == 0 ? 2 : 1); }

static int mean_patch_blocks(int n1, int n2, int n3, int vz) {
  const long nch = (long)n1 * n2 * (n3 / vz);
  long nb = (nch + kThreads - 1) / kThreads;
  if (nb > kPatchBlocks) nb = kPatchBlocks;
  return (int)(nb < 1 ? 1 : nb);
}

size_t mean_patch_workspace(int /*dtype*/, int C, int n1, int n2, int n3) {
  return (size_t)mean_patch_blocks(n1, n2, n3, mean_patch_vz(n3)) * 27 * C * sizeof(double);
}

template <typename TI>
static void launch_mp_t(const void* img, double* part, int nblk, bool one, double invV, const void* w0,
                        const void* b0, void* z0, const void* w1, const void* b1, void* z1, void* ybar, int C, int n1,
                        int n2, int n3, int vz, hipStream_t st) {
  typedef typename AccOf<TI>::type A;
#define MLPCG_MP(CC, VZZ)                                                                                        \
  if (C == CC && vz == VZZ) {                                                                                    \
    if (one) {                                                                                                   \
      mean_patch_one_kernel<TI, CC, VZZ><<<1, kPatchFinalThreads, 0, st>>>(                                      \
          (const TI*)img, n1, n2, n3, invV, (const A*)w0, (const A*)b0, (A*)z0, (const A*)w1, (const A*)b1, (A*)z1, \
          (A*)ybar);                                                                                             \
    } else {                                                                                                     \
      mean_patch_partial_kernel<TI, CC, VZZ><<<nblk, kThreads, 0, st>>>((const TI*)img, n1, n2, n3, part);       \
      mean_patch_final_kernel<A><<<1, kPatchFinalThreads, 0, st>>>(part, nblk, n1, n2, n3, 27 * C, invV,         \
                                                                   (const A*)w0, (const A*)b0, (A*)z0,           \
                                                                   (const A*)w1, (const A*)b1, (A*)z1, (A*)ybar); \
    }                                                                                                            \
    return;                                                                                                      \
  }
  MLPCG_MP(1, 4) MLPCG_MP(1, 2) MLPCG_MP(1, 1)
  MLPCG_MP(2, 4) MLPCG_MP(2, 2) MLPCG_MP(2, 1)
  MLPCG_MP(3, 4) MLPCG_MP(3, 2) MLPCG_MP(3, 1)
#undef MLPCG_MP
}

int launch_sm_linear_pair(int dtype, const void* img, const void* w0, const void* b0, void* z0,
                          const void* w1, const void* b1, void* z1, void* ybar, void* workspace, int C,
                          int n1, int n2, int n3, hipStream_t st) {
  MLPCG_REQUIRE(C >= 1 && C <= 3, "sm_linear: C must be 1, 2 or 3 (got %d)", C);
  MLPCG_REQUIRE(!w1 || (b1 && z1), "sm_linear: a second weight needs its bias and output");
  const int vz = mean_patch_vz(n3);
  const int nblk = mean_patch_blocks(n1, n2, n3, vz);
  double* part = (double*)workspace;
  const double invV = 1.0 / ((double)n1 * n2 * n3);
  const bool one = (long)n1 * n2 * (n3 / vz) <= kPatchOneRuns;
#define MLPCG_MPT(T) launch_mp_t<T>(img, part, nblk, one, invV, w0, b0, z0, w1, b1, z1, ybar, C, n1, n2, n3, vz, st)
  switch (dtype) {
    case kF64: MLPCG_MPT(double); break;
    case kF32: MLPCG_MPT(float); break;
    case kF16: MLPCG_MPT(f16); break;
    case kBF16: MLPCG_MPT(bf16); break;
    default: MLPCG_REQUIRE(false, "sm_linear: bad dtype %d", dtype);
  }
#undef MLPCG_MPT
  return check_launch("sm_linear");
}

int launch_sm_linear(int dtype, const void* img, const void* w, const void* b, void* z, void* ybar,
                     void* workspace, int C, int n1, int n2, int n3, hipStream_t st) {
  return launch_sm_linear_pair(dtype, img, w, b, z, nullptr, nullptr, nullptr, ybar, workspace, C, n1, n2, n3,
                               st);
}

// ---------------------------------------------------------------------------
// SM linear without allocation.  The block partials of the mean patch go to a file-scope
// device array instead of a caller workspace: at most 1024 blocks x 27 C doubles
// (648 KiB for C = 3) for ANY grid, since the partial kernel caps its block count (at half of that).
// Each GPU holds its own copy of the array until the process ends; host code never
// passes the array's name to a kernel (in host code it names a host-side stand-in) but
// the device address that hipGetSymbolAddress returned, fetched once per device with
// that device current.  Calls that overlap on one GPU share the array and race; nothing
// in it needs clearing (every launched block writes all of its partials before the
// final pass reads them).
// ---------------------------------------------------------------------------
constexpr size_t kScratchBytes = (size_t)1024 * 27 * 3 * sizeof(double);
static __device__ __align__(256) double scratch[kScratchBytes / sizeof(double)];

constexpr int kMaxScratchDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxScratchDevices] = {};

size_t sm_linear_scratch_bytes() { return kScratchBytes; }

static int scratch_for_current_device(void** out) {
  int dev = -1;
  MLPCG_HIP(hipGetDevice(&dev));
  MLPCG_REQUIRE(dev >= 0 && dev < kMaxScratchDevices, "sm_linear_noalloc: device %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    MLPCG_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    MLPCG_REQUIRE(p != nullptr, "sm_linear_noalloc: no device address for the scratch array");
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

int launch_sm_linear_noalloc(int dtype, const void* img, const void* w, const void* b, void* z, void* ybar,
                             int C, int n1, int n2, int n3, hipStream_t st) {
  MLPCG_REQUIRE(C >= 1 && C <= 3, "sm_linear_noalloc: C must be 1, 2 or 3 (got %d)", C);
  MLPCG_REQUIRE(n1 >= 1 && n2 >= 1 && n3 >= 1, "sm_linear_noalloc: bad grid (%d,%d,%d)", n1, n2, n3);
  const size_t need = mean_patch_workspace(dtype, C, n1, n2, n3);
  MLPCG_REQUIRE(need <= kScratchBytes,
                "sm_linear_noalloc: the reduction needs %zu bytes of scratch, more than the %zu reserved", need,
                kScratchBytes);
  void* ws = nullptr;
  if (scratch_for_current_device(&ws)) return -1;
  return launch_sm_linear(dtype, img, w, b, z, ybar, ws, C, n1, n2, n3, st);
}

// gw = g * ybar, gb = g  (sm_linear_3d_kernel.cu:229-238)
template <typename A>
__global__ void linear_backward_kernel(const A* __restrict__ g, const A* __restrict__ ybar,
                                       A* __restrict__ gw, A* __restrict__ gb, int NV) {
  const A gv = g[0];
  for (int o = threadIdx.x; o < NV; o += blockDim.x) gw[o] = gv * ybar[o];
  if (threadIdx.x == 0) gb[0] = gv;
}

int launch_linear_backward(int dtype, const void* g, const void* ybar, void* gw, void* gb, int C,
                           hipStream_t st) {
  if (dtype == kF64)
    linear_backward_kernel<double><<<1, 128, 0, st>>>((const double*)g, (const double*)ybar,
                                                      (double*)gw, (double*)gb, 27 * C);
  else
    linear_backward_kernel<float><<<1, 128, 0, st>>>((const float*)g, (const float*)ybar, (float*)gw,
                                                     (float*)gb, 27 * C);
  return check_launch("sm_linear_backward");
}

// ---------------------------------------------------------------------------
// Weight gradient.
// ---------------------------------------------------------------------------
template <int C> struct WGShape {
  static constexpr int NQ = 27 * C + 1;          // patch columns + bias column
  static constexpr int RP = 3, RQ = 4;           // register tile
  static constexpr int NPG = 9;                  // 27 / RP
  static constexpr int NQG = (NQ + RQ - 1) / RQ;
  static constexpr int NQP = NQG * RQ;           // padded patch rows in LDS
  static constexpr int NT = NPG * NQG;           // threads per voxel subset
  static constexpr int NSUB = kThreads / NT;     // voxel subsets
  static constexpr int NO = 27 * NQ;             // outputs
};

template <typename TX, typename TI, int C, int TV>
__global__ __launch_bounds__(kThreads) void weight_grad_partial_kernel(
    const TX* __restrict__ a, const TX* __restrict__ cv, int B, const TI* __restrict__ img, int n1,
    int n2, int n3, typename AccOf<TX>::type* __restrict__ partials) {
  typedef typename AccOf<TX>::type A;
  typedef WGShape<C> S;
  constexpr int LD = TV + 1;
  __shared__ A Gs[27 * LD];
  __shared__ A Ps[S::NQP * LD];
  static_assert(S::NSUB >= 1, "tile too large");
  static_assert(27 * LD >= kThreads * S::RP * S::RQ, "reduction buffer too small");
  const int tid = threadIdx.x;
  const int tile_id = tid % S::NT, sub = tid / S::NT;
  const int pg = tile_id / S::NQG, qg = tile_id % S::NQG;
  const long V = (long)n1 * n2 * n3;
  const long s1 = (long)n2 * n3;
  A acc[S::RP][S::RQ];
#pragma unroll
  for (int r = 0; r < S::RP; ++r)
#pragma unroll
    for (int q = 0; q < S::RQ; ++q) acc[r][q] = A(0);
  for (int r = S::NQ; r < S::NQP; ++r)
    for (int u = tid; u < TV; u += kThreads) Ps[r * LD + u] = A(0);

  const long ntiles = (V + TV - 1) / TV;
  for (long tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    if (tid < TV) {
      const long v = tile * TV + tid;
      A G[27];
      A P[27 * C];
#pragma unroll
      for (int p = 0; p < 27; ++p) G[p] = A(0);
#pragma unroll
      for (int q = 0; q < 27 * C; ++q) P[q] = A(0);
      if (v < V) {
        const int k = (int)(v % n3);
        const int j = (int)((v / n3) % n2);
        const int i = (int)(v / s1);
        bool in[27];
        long off[27];
#pragma unroll
        for (int p = 0; p < 27; ++p) {
          const int d1 = p / 9 - 1, d2 = (p / 3) % 3 - 1, d3 = p % 3 - 1;
          in[p] = (unsigned)(i + d1) < (unsigned)n1 && (unsigned)(j + d2) < (unsigned)n2 &&
                  (unsigned)(k + d3) < (unsigned)n3;
          off[p] = d1 * s1 + (long)d2 * n3 + d3;
        }
        for (int b = 0; b < B; ++b) {
          const A av = (A)a[(long)b * V + v];
          const TX* cb = cv + (long)b * V + v;
#pragma unroll
          for (int p = 0; p < 27; ++p)
            if (in[p]) G[p] += av * (A)cb[off[p]];
        }
#pragma unroll
        for (int s = 0; s < C; ++s)
#pragma unroll
          for (int p = 0; p < 27; ++p)
            if (in[p]) P[s * 27 + p] = (A)img[s * V + v + off[p]];
      }
#pragma unroll
      for (int p = 0; p < 27; ++p) Gs[p * LD + tid] = G[p];
#pragma unroll
      for (int q = 0; q < 27 * C; ++q) Ps[q * LD + tid] = P[q];
      Ps[(27 * C) * LD + tid] = (v < V) ? A(1) : A(0);
    }
    __syncthreads();
    if (sub < S::NSUB) {
      for (int u = sub; u < TV; u += S::NSUB) {
        A g[S::RP], pv[S::RQ];
#pragma unroll
        for (int r = 0; r < S::RP; ++r) g[r] = Gs[(pg * S::RP + r) * LD + u];
#pragma unroll
        for (int q = 0; q < S::RQ; ++q) pv[q] = Ps[(qg * S::RQ + q) * LD + u];
#pragma unroll
        for (int r = 0; r < S::RP; ++r)
#pragma unroll
          for (int q = 0; q < S::RQ; ++q) acc[r][q] += g[r] * pv[q];
      }
    }
    __syncthreads();
  }
  A* red = Gs;
  if (sub < S::NSUB) {
#pragma unroll
    for (int r = 0; r < S::RP; ++r)
#pragma unroll
      for (int q = 0; q < S::RQ; ++q)
        red[((sub * S::NT + tile_id) * S::RP + r) * S::RQ + q] = acc[r][q];
  }
  __syncthreads();
  if (tid < S::NT) {
#pragma unroll
    for (int r = 0; r < S::RP; ++r) {
#pragma unroll
      for (int q = 0; q < S::RQ; ++q) {
        A s = A(0);
        for (int sb = 0; sb < S::NSUB; ++sb) s += red[((sb * S::NT + tile_id) * S::RP + r) * S::RQ + q];
        const int op = pg * S::RP + r, oq = qg * S::RQ + q;
        if (oq < S::NQ) partials[(size_t)blockIdx.x * S::NO + op * S::NQ + oq] = s;
      }
    }
  }
}

// BF16 weight gradient on the BF16 matrix cores (v_mfma_f32_16x16x32_bf16), B == 1,
// n3 % 64 == 0, any C <= 3.  G_p(v) = a(v) c(v + d_p) of two BF16 values has at most 16
// significant bits, so it is exact in FP32 and splits exactly into hi + lo BF16 parts
// (hi: the top 8 bits by truncation, lo = G - hi: the remaining <= 8 bits).  With
// D[p][q] = sum_v hi_p(v) P_q(v) + lo_p(v) P_q(v) every product is exact and the sums are
// FP32, as in the FP32-operand kernels above; the matrix cores do 32 voxels per product
// instead of 4.
//
// A wave walks a column of z-row segments (plane i, rows j0 .. j0 + J - 1, 64 z cells,
// two K chunks of 32 voxels) and keeps the three neighbour rows along j of each plane
// i - 1, i, i + 1 in a ring of LDS slots, so each step stages one new row per plane
// (loaded into registers during the previous step's products).  x rows are stored as FP32
// (one copy; a lane's 8 taps along z are read at 4-byte alignment), image rows as three
// BF16 copies shifted by one cell so that every B operand is one aligned 16-byte read.
// Operand layout: A[p][k] lane 16 kb + m holds row m, voxels kv .. kv + 7 of the chunk with
// kv = 16 (kb & 1) + 8 (kb >> 1); B[k][q] lane 16 kb + m holds column m of the same voxels;
// D[4 kb + i][m].  Rows p = 27..31 and columns q > 27C read constant zero rows, column 27C
// (bias) a row of ones.  LDS banks (32 x 4 bytes, 32 lanes per cycle): the two lane groups
// of a half-wave read x words 16 apart, and the x rows of a ring (slot pitch kXP, plane
// pitch kXPP words) start at offsets that keep the 16 taps of a half-wave on distinct
// banks mod 16 for most ring positions (a CPU model of the x-operand reads: 107 LDS cycles
// per step, 64 without conflicts, against 213 with the lane groups' voxels side by side and
// 72-word rows).
namespace wgb {
constexpr int kSeg = 64;                       // z cells per row segment
constexpr int kXS = 72;                        // FP32 zero row length; x row: cell z0 - 1 + e at element 3 + e
constexpr int kXP = 70, kXPP = 212;            // x ring: slot and plane pitch (words)
constexpr int kXW = 2 * kXPP + 2 * kXP + 72;   // x ring words per wave
constexpr int kIS = 72;                        // BF16 image row copy (64 cells used)
constexpr int kXBytes = 4 * kXW * 4;           // x rings of the 4 waves
constexpr int kGBytes = 4 * kSeg * 4;          // a rows (FP32) of the 4 waves
constexpr int kZBytes = kXS * 4;               // FP32 zero row
constexpr int kCBytes = 2 * kIS * 2;           // BF16 zero row, ones row
__host__ __device__ constexpr int img_bytes(int C) { return 4 * C * 27 * kIS * 2; }
__host__ __device__ constexpr int lds_bytes(int C) { return kXBytes + kGBytes + kZBytes + kCBytes + img_bytes(C); }
}  // namespace wgb

typedef __bf16 wg_bf16x8 __attribute__((ext_vector_type(8), aligned(16)));
typedef uint32_t wg_u32x4 __attribute__((ext_vector_type(4)));

// hi / lo BF16 parts of an exact FP32 product, packed in pairs (element 0 in the low half)
__device__ __forceinline__ void wg_split2(float p0, float p1, uint32_t& hi, uint32_t& lo) {
  const uint32_t u0 = __float_as_uint(p0), u1 = __float_as_uint(p1);
  const float l0 = p0 - __uint_as_float(u0 & 0xffff0000u);
  const float l1 = p1 - __uint_as_float(u1 & 0xffff0000u);
  hi = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
  lo = __builtin_amdgcn_perm(__float_as_uint(l1), __float_as_uint(l0), 0x07060302u);
}

template <int C>
__global__ __launch_bounds__(kThreads) void weight_grad_bf16_kernel(
    const bf16* __restrict__ a, const bf16* __restrict__ cv, const bf16* __restrict__ img, int n1,
    int n2, int n3, int J, float* __restrict__ partials) {
  using namespace wgb;
  constexpr int NQ = 27 * C + 1, NT = (NQ + 15) / 16, NO = 27 * NQ;
  constexpr int NTASK = 24 + 24 * C + 8, NR = (NTASK + 63) / 64;  // staging tasks per step
  static_assert(4 * 27 * NQ * 4 <= img_bytes(C), "reduction buffer");
  __shared__ __attribute__((aligned(16))) char lds[lds_bytes(C)];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int m = lane & 15, kb = lane >> 4;
  // byte offsets in lds
  const int oX = w * kXW * 4;
  const int kv = ((kb & 1) << 4) | ((kb >> 1) << 3);  // first voxel of the lane's 8 in a chunk
  const int oG = kXBytes + w * kSeg * 4;
  const int oZ = kXBytes + kGBytes;
  const int oC = oZ + kZBytes;
  const int oI = oC + kCBytes + w * C * 27 * kIS * 2;
  for (int e = threadIdx.x; e < kXS; e += kThreads) *(float*)(lds + oZ + 4 * e) = 0.f;
  for (int e = threadIdx.x; e < 2 * kIS; e += kThreads)
    *(uint16_t*)(lds + oC + 2 * e) = e < kIS ? (uint16_t)0 : (uint16_t)0x3f80;  // BF16 0, 1
  __syncthreads();

  // this lane's operand rows: A taps p = 16 h + m, B columns q = 16 gt + m.  Offset at
  // step j = base + slot * stride with slot = (j + 2 + e2) mod 3 the ring slot of row
  // j + e2 - 1 (e2 = d2 + 1); constant rows have stride 0.
  int abase[2], ae2[2], astr[2], bbase[NT], be2[NT], bstr[NT];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int p = 16 * h + m;
    if (p < 27) {
      abase[h] = oX + ((p / 9) * kXPP + 3 + p % 3 + kv) * 4;
      ae2[h] = (p / 3) % 3;
      astr[h] = kXP * 4;
    } else {
      abase[h] = oZ + kv * 4;
      ae2[h] = 0;
      astr[h] = 0;
    }
  }
#pragma unroll
  for (int gt = 0; gt < NT; ++gt) {
    const int q = 16 * gt + m;
    if (q < 27 * C) {
      const int c = q / 27, s = q % 27;
      bbase[gt] = oI + (((c * 9 + (s / 9) * 3) * 3 + s % 3) * kIS + kv) * 2;
      be2[gt] = (s / 3) % 3;
      bstr[gt] = 3 * kIS * 2;
    } else {
      bbase[gt] = oC + ((q == 27 * C ? kIS : 0) + kv) * 2;
      be2[gt] = 0;
      bstr[gt] = 0;
    }
  }

  const long V = (long)n1 * n2 * n3;
  const int nseg3 = n3 / kSeg, njb = (n2 + J - 1) / J;
  const long ncol = (long)n1 * nseg3 * njb;
  typedef float f4 __attribute__((ext_vector_type(4)));
  f4 acc[2][NT];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int gt = 0; gt < NT; ++gt) acc[h][gt] = f4{0.f, 0.f, 0.f, 0.f};

  // staging task e of a step: e < 24: x row (plane i + e / 8 - 1, row jr), chunk e % 8;
  // e < 24 + 24C: image channel, same rows; else the a row (i, ja), chunk e % 8.  A task
  // loads the chunk's 8 cells plus the cell pairs before and after it (zero outside the grid).
  struct Regs {
    uint32_t d[NR][6];
  };
  auto task_src = [&](int e, int i, int jr, int ja, int z0, const bf16*& src, bool& ok, int& t) {
    int ii, jj;
    if (e < 24) {
      src = cv;
      ii = i + e / 8 - 1;
      jj = jr;
    } else if (e < 24 + 24 * C) {
      const int f = e - 24;
      src = img + (long)(f / 24) * V;
      ii = i + (f % 24) / 8 - 1;
      jj = jr;
    } else {
      src = a;
      ii = i;
      jj = ja;
    }
    t = e & 7;
    ok = e < NTASK && (unsigned)ii < (unsigned)n1 && (unsigned)jj < (unsigned)n2;
    src += ((long)(ok ? ii : 0) * n2 + (ok ? jj : 0)) * n3 + z0 + 8 * t;
  };
  auto load_step = [&](Regs& r, int i, int jr, int ja, int z0) {
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int e = lane + 64 * k;
      const bf16* src;
      bool ok;
      int t;
      task_src(e, i, jr, ja, z0, src, ok, t);
      const uint32_t* s32 = (const uint32_t*)src;
      const wg_u32x4 v = ok ? *(const wg_u32x4*)s32 : wg_u32x4{0u, 0u, 0u, 0u};
      const bool okp = ok && z0 + 8 * t > 0, okn = ok && z0 + 8 * t + 8 < n3;
      r.d[k][0] = okp ? s32[-1] : 0u;
      r.d[k][1] = v[0];
      r.d[k][2] = v[1];
      r.d[k][3] = v[2];
      r.d[k][4] = v[3];
      r.d[k][5] = okn ? s32[4] : 0u;
    }
  };
  // slot of row jr in the ring: (jr + 3) mod 3 (jr >= -1)
  auto write_step = [&](const Regs& r, int jr) {
    const int sl = (jr + 3) % 3;
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int e = lane + 64 * k;
      const int t = e & 7;
      const uint32_t* d = r.d[k];
      if (e < 24) {
        // rows start at even words (8-byte stores)
        char* dst = lds + oX + ((e / 8) * kXPP + sl * kXP + 4 + 8 * t) * 4;
        typedef float f2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int u = 0; u < 4; ++u)
          *(f2*)(dst + 8 * u) = f2{__uint_as_float(d[1 + u] << 16), __uint_as_float(d[1 + u] & 0xffff0000u)};
        if (t == 0) *(float*)(dst - 4) = __uint_as_float(d[0] & 0xffff0000u);
        if (t == 7) *(float*)(dst + 32) = __uint_as_float(d[5] << 16);
      } else if (e < 24 + 24 * C) {
        const int f = e - 24;
        char* dst = lds + oI + ((((f / 24) * 9 + ((f % 24) / 8) * 3 + sl) * 3) * kIS + 8 * t) * 2;
        *(wg_u32x4*)dst = wg_u32x4{__builtin_amdgcn_alignbyte(d[1], d[0], 2), __builtin_amdgcn_alignbyte(d[2], d[1], 2),
                                   __builtin_amdgcn_alignbyte(d[3], d[2], 2), __builtin_amdgcn_alignbyte(d[4], d[3], 2)};
        *(wg_u32x4*)(dst + kIS * 2) = wg_u32x4{d[1], d[2], d[3], d[4]};
        *(wg_u32x4*)(dst + 2 * kIS * 2) =
            wg_u32x4{__builtin_amdgcn_alignbyte(d[2], d[1], 2), __builtin_amdgcn_alignbyte(d[3], d[2], 2),
                     __builtin_amdgcn_alignbyte(d[4], d[3], 2), __builtin_amdgcn_alignbyte(d[5], d[4], 2)};
      } else if (e < NTASK) {
        char* dst = lds + oG + 8 * t * 4;
        *(f4*)dst = f4{__uint_as_float(d[1] << 16), __uint_as_float(d[1] & 0xffff0000u),
                       __uint_as_float(d[2] << 16), __uint_as_float(d[2] & 0xffff0000u)};
        *(f4*)(dst + 16) = f4{__uint_as_float(d[3] << 16), __uint_as_float(d[3] & 0xffff0000u),
                              __uint_as_float(d[4] << 16), __uint_as_float(d[4] & 0xffff0000u)};
      }
    }
  };
  auto wave_sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  for (long col = (long)blockIdx.x * 4 + w; col < ncol; col += (long)gridDim.x * 4) {
    // column order: plane fastest, so the waves of a block share neighbour planes
    const int i = (int)(col % n1);
    const long rest = col / n1;
    const int jb = (int)(rest % njb);
    const int z0 = (int)(rest / njb) * kSeg;
    const int j0 = jb * J, j1 = min(j0 + J, n2);
    Regs r;
    // prologue: rows j0 - 1 and j0 (the a-row tasks of these two are not used)
    load_step(r, i, j0 - 1, j0, z0);
    write_step(r, j0 - 1);
    load_step(r, i, j0, j0, z0);
    write_step(r, j0);
    load_step(r, i, j0 + 1, j0, z0);
    for (int j = j0; j < j1; ++j) {
      write_step(r, j + 1);  // row j + 1 and the a row of j
      wave_sync();
      if (j + 1 < j1) load_step(r, i, j + 2, j + 1, z0);
      const int sj = (j + 2) % 3;
      int ao[2], bo[NT];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        int s = sj + ae2[h];
        s = s >= 3 ? s - 3 : s;
        ao[h] = abase[h] + s * astr[h];
      }
#pragma unroll
      for (int gt = 0; gt < NT; ++gt) {
        int s = sj + be2[gt];
        s = s >= 3 ? s - 3 : s;
        bo[gt] = bbase[gt] + s * bstr[gt];
      }
#pragma unroll
      for (int cc = 0; cc < 2; ++cc) {
        const f4 g0 = *(const f4*)(lds + oG + (32 * cc + kv) * 4);
        const f4 g1 = *(const f4*)(lds + oG + (32 * cc + kv + 4) * 4);
        const float gv[8] = {g0[0], g0[1], g0[2], g0[3], g1[0], g1[1], g1[2], g1[3]};
        wg_bf16x8 ahi[2], alo[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float* xp = (const float*)(lds + ao[h] + 128 * cc);
          uint32_t hi[4], lo[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) wg_split2(gv[2 * k] * xp[2 * k], gv[2 * k + 1] * xp[2 * k + 1], hi[k], lo[k]);
          ahi[h] = __builtin_bit_cast(wg_bf16x8, wg_u32x4{hi[0], hi[1], hi[2], hi[3]});
          alo[h] = __builtin_bit_cast(wg_bf16x8, wg_u32x4{lo[0], lo[1], lo[2], lo[3]});
        }
#pragma unroll
        for (int gt = 0; gt < NT; ++gt) {
          const wg_bf16x8 bv = *(const wg_bf16x8*)__builtin_assume_aligned(lds + bo[gt] + 64 * cc, 16);
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            acc[h][gt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ahi[h], bv, acc[h][gt], 0, 0, 0);
            acc[h][gt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(alo[h], bv, acc[h][gt], 0, 0, 0);
          }
        }
      }
      wave_sync();
    }
  }
  // D[16 h + 4 kb + t][16 gt + m] of this wave -> LDS (over the image slots), then a
  // fixed-order sum over the four waves
  __syncthreads();
  float* red = (float*)(lds + kXBytes + kGBytes + kZBytes + kCBytes);
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int gt = 0; gt < NT; ++gt)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int p = 16 * h + 4 * kb + t, q = 16 * gt + m;
        if (p < 27 && q < NQ) red[(w * 27 + p) * NQ + q] = acc[h][gt][t];
      }
  __syncthreads();
  for (int o = threadIdx.x; o < NO; o += kThreads)
    partials[(size_t)blockIdx.x * NO + o] = (red[o] + red[NO + o]) + (red[2 * NO + o] + red[3 * NO + o]);
}

template <typename A>
__global__ __launch_bounds__(kThreads) void weight_grad_final_kernel(const A* __restrict__ partials,
                                                                     int nblk, int C,
                                                                     A* __restrict__ gW,
                                                                     A* __restrict__ gb) {
  // one block per output; the block sums the nblk partials (strided, then block-reduced)
  __shared__ double sh[4];
  const int NQ = 27 * C + 1, NO = 27 * NQ;
  const int o = blockIdx.x;
  if (o >= NO) return;
  double s = 0.0;
  for (int blk = threadIdx.x; blk < nblk; blk += kThreads) s += (double)partials[(size_t)blk * NO + o];
  s = block_sum(s, sh);
  if (threadIdx.x != 0) return;
  const int p = o / NQ, q = o % NQ;
  if (q < 27 * C) gW[p * 27 * C + q] = (A)s;
  else gb[p] = (A)s;
}

static int wg_tv(int dtype, int C) { return (dtype == kF64 && C >= 2) ? 128 : 256; }

static int wg_blocks(int dtype, int C, int n1, int n2, int n3) {
  const long V = (long)n1 * n2 * n3;
  const int tv = wg_tv(dtype, C);
  long nb = (V + tv - 1) / tv;
  if (nb > 1024) nb = 1024;
  return (int)(nb < 1 ? 1 : nb);
}

size_t weight_grad_workspace(int dtype, int C, int /*B*/, int n1, int n2, int n3) {
  const size_t acc = dtype == kF64 ? sizeof(double) : sizeof(float);
  return (size_t)wg_blocks(dtype, C, n1, n2, n3) * 27 * (27 * C + 1) * acc;
}

int launch_weight_grad(int dtype, const void* a, const void* c, const void* img, void* gW, void* gb,
                       void* workspace, int C, int B, int n1, int n2, int n3, hipStream_t st) {
  MLPCG_REQUIRE(C >= 1 && C <= 3, "weight_grad: C must be 1, 2 or 3 (got %d)", C);
  const int nblk = wg_blocks(dtype, C, n1, n2, n3);
  const int NO = 27 * (27 * C + 1);
  if (dtype == kF64) {
    const double *pa = (const double*)a, *pc = (const double*)c, *pi = (const double*)img;
    double* part = (double*)workspace;
    if (C == 1) weight_grad_partial_kernel<double, double, 1, 256><<<nblk, kThreads, 0, st>>>(pa, pc, B, pi, n1, n2, n3, part);
    else if (C == 2) weight_grad_partial_kernel<double, double, 2, 128><<<nblk, kThreads, 0, st>>>(pa, pc, B, pi, n1, n2, n3, part);
    else weight_grad_partial_kernel<double, double, 3, 128><<<nblk, kThreads, 0, st>>>(pa, pc, B, pi, n1, n2, n3, part);
    weight_grad_final_kernel<double><<<NO, kThreads, 0, st>>>(part, nblk, C, (double*)gW, (double*)gb);
    return check_launch("weight_grad");
  }
  float* part = (float*)workspace;
  int nb = nblk;
  if (dtype == kBF16 && B == 1 && n3 % wgb::kSeg == 0) {
    // whole 64-cell segments of one BF16 right-hand side: columns of J segments, about one
    // column per wave, with ring staging (256^3 C = 1 134 to 157 us from box to box, C = 3 240
    // to 250, against 190 and 480 us of the tiles below with FP32 data)
    const long segs = (long)n1 * n2 * (n3 / wgb::kSeg);
    const long per_wave = (segs + 4L * nblk - 1) / (4L * nblk);
    const int J = (int)(per_wave < 4 ? 4 : (per_wave > 64 ? 64 : per_wave));
    const bf16 *pa = (const bf16*)a, *pc = (const bf16*)c, *pi = (const bf16*)img;
    if (C == 1) weight_grad_bf16_kernel<1><<<nblk, kThreads, 0, st>>>(pa, pc, pi, n1, n2, n3, J, part);
    else if (C == 2) weight_grad_bf16_kernel<2><<<nblk, kThreads, 0, st>>>(pa, pc, pi, n1, n2, n3, J, part);
    else weight_grad_bf16_kernel<3><<<nblk, kThreads, 0, st>>>(pa, pc, pi, n1, n2, n3, J, part);
  } else {
    nb = wgrad_blocks(nblk, n1, n2, n3);
    const int e = launch_wgrad(dtype, a, c, img, part, nb, C, B, n1, n2, n3, st);
    if (e) return e;
  }
  weight_grad_final_kernel<float><<<NO, kThreads, 0, st>>>(part, nb, C, (float*)gW, (float*)gb);
  return check_launch("weight_grad");
}

}  // namespace mlpcg
