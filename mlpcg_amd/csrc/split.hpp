// FP32 SM block on the matrix cores, by FP16 operands split in two.
//
//   y[b, v] = sum_p K_p(v) x[b, v + d_p],   K_p(v) = b_p + sum_{c,s} W[p,c,s] img[c, v + d_s]
//
// (sm_block_3d_kernel.cu:46-70), all in FP32.  K is neither stored nor streamed (108 of the
// 116 bytes per voxel of the stored-stencil apply): it is recomputed from the image tile in
// LDS.  W and the image are scaled by powers of two and split as v = hi + lo into two FP16
// values each, which keeps 22 bits and more, and
//   W . img = W_lo img_hi + W_hi img_lo + W_hi img_hi          (FP16 products, FP32 sums)
// on v_mfma_f32_32x32x16_f16, the small products first.  The dropped W_lo img_lo is below 2^-22
// of its term, the matrix cores round a few times where an FP32 chain rounds 28 times; measured
// against 64 bits the block's error is below that of the FP32 chain (see launch_sm_split).  K
// meets x in FP32 FMAs.
//
// Scaling.  A channel of W is scaled to a largest value in [2^14, 2^15) when it is packed, a
// channel of a workgroup's image tile likewise, less what makes all products share one unit
// 2^-E: the channel whose W times image is largest decides, and the bias, which joins scaled by
// 2^E as three FP16 parts (33 bits) on spare K slots whose image value is 2^15 (as an
// accumulator it took 16 registers and a wave per SIMD).  y is scaled back once.  FP16's smallest
// step 2^-24 is then 2^-39 of the largest value: what is within 2^-16 of that keeps its bits.
//
// Exact stencils.  Where more is asked for, K comes from FP32 FMAs over the image as it is (some
// ten times slower): blocks with infinite or NaN weights or whose weights along a line of three
// taps are all, but not all 0, below 2^-16 of their channel's largest; tiles with an infinite or
// NaN image value, with three image cells in a row like that (of what the tile's scaling
// leaves), or with |x| from 2^80 on, which the unscaled K alone can take without overflow.
//
// Tile and lanes.  A workgroup of 4 waves covers FI planes x 8 rows x 64 z; the tile with a
// one-cell halo is staged in LDS (x in FP32, the image as two FP16 arrays), zero outside the
// grid, so any extents are taken.  A wave takes one row of 64 voxels at a time (a chunk) as
// two groups of 32 of one z parity: lane (h, n) = (lane / 32, lane % 32) works on voxels
// z = 2n and 2n + 1.  The 27 taps, as 9 columns (d1, d2) of three, go to the two lane
// halves, columns 0..4 and 6, 7, 8, 5: per column the two aligned words w0 = cells 2n - 1, 2n and
// w1 = 2n + 1, 2n + 2 hold all three taps of both voxels.
// Operands (lane l, element j / i): A[l % 32][8 (l / 32) + j], B[8 (l / 32) + j][l % 32],
// D[8 (i / 4) + 4 (l / 32) + i % 4][l % 32].  A = W, B = image patches; the rows of D are
// ordered so that a lane receives K of its own columns' taps, register i = tap 3 (i / 3) +
// i % 3 of its five columns, and dots them with the x it reads itself; one 32-lane swap adds
// the halves.  The K slots of a lane are its columns' words as they lie (w0 for even
// voxels: taps -1, 0; w1 for odd: taps 0, +1), then the third taps, packed from the halves
// of the other words.
//
// Tiles whose image is exact in one FP16 value (flags, fluid interiors) leave img_lo out;
// tiles of zero x, and chunks that the output mask zeroes, skip their products.
#pragma once

#include "kernels.hpp"
#include "split_common.hpp"

namespace mlpcg {
namespace split {

constexpr int kZ = 64, kJ = 8, kPJ = kJ + 2;
constexpr int kPitch = 68;      // cells per staged row (66 used; even, for 8-byte x reads)
constexpr int kTarget = 14;  // largest |W| and |img| of a channel are scaled into [2^14, 2^15)
constexpr int kOne = 15;     // exponent of the image value of the bias's slots
constexpr float kHuge = 1.2089258e24f;  // 2^80


// column i (0..4) of lane half h; the fifth of the upper half is a dummy (zero weights).  The
// first three are a plane's (d1 = -1, +1), which the input gradient (igrad.hpp) relies on.
__host__ __device__ constexpr int col_of(int h, int i) { return h == 0 ? i : (i < 3 ? 6 + i : i == 3 ? 5 : 8); }
__host__ __device__ constexpr bool col_real(int h, int i) { return h == 0 || i < 4; }

struct PackHeader {
  int w_exp[3];     // exponents of the channels' factors (kNone: no weight but 0)
  int bias_limit;   // largest E that the bias leaves
  int finite;       // no weight or bias is infinite or NaN
  int exact;        // two FP16 values do not hold the weights
};
constexpr int kNone = 1000;
// header, then W [parity][hi, lo][k half][channel][lane][8] (FP16), the bias of the 32 rows of D,
// and W as it is, in the order of a lane's results: [27 C taps, bias][lane half][16] (FP32)
constexpr size_t kHeaderBytes = 64;
constexpr size_t pack_w_bytes(int C) { return (size_t)2 * 2 * 2 * C * 64 * 8 * sizeof(f16); }
constexpr size_t pack_exact_at(int C) { return kHeaderBytes + pack_w_bytes(C) + 32 * sizeof(float); }
constexpr size_t pack_bytes(int C) { return pack_exact_at(C) + (size_t)(27 * C + 1) * 32 * sizeof(float); }

// Tap (of 27) of K slot j of lane half h in k half kc for z parity par; -1: spare.
__host__ __device__ constexpr int slot_tap(int par, int h, int kc, int j) {
  const int w = 4 * kc + j / 2, hf = j & 1;
  const int third = par == 0 ? 2 : 0;  // the tap outside the aligned pair
  const int i = w < 5 ? w : w == 5 ? hf : w == 6 ? 2 + hf : 4;
  const int a3 = w < 5 ? (par == 0 ? hf : 1 + hf) : third;
  if (w == 7 && hf != (par == 0 ? 0 : 1)) return -1;
  return col_real(h, i) ? 3 * col_of(h, i) + a3 : -1;
}
// the spare slot (of k half 1)
__host__ __device__ constexpr int spare_slot(int par) { return par == 0 ? 7 : 6; }
// Tap of result register i of lane half h; -1: none.
__host__ __device__ constexpr int reg_tap(int h, int i) {
  return i < 15 && col_real(h, i / 3) ? 3 * col_of(h, i / 3) + i % 3 : -1;
}

// One workgroup per 512 packed values; every workgroup scans the weights for their scale.
__global__ __launch_bounds__(kThreads) void split_pack_kernel(const float* __restrict__ W, const float* __restrict__ b,
                                                              int C, char* __restrict__ out) {
  __shared__ unsigned sh[5][4];
  unsigned mw[3] = {0, 0, 0}, mb = 0, bad = 0, line[3];
  int lc[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {  // lines of three taps (C <= 3; clamped, so that all loads are in flight together)
    const int t = min(k * kThreads + (int)threadIdx.x, 243 * C - 1);
    lc[k] = t / 9 % C;
    float m = 0.f;
#pragma unroll
    for (int u = 0; u < 3; ++u) m = max_nan(m, fabsf(W[3 * t + u]));
    bad |= magnitude(m) >= kInfinity;
    line[k] = magnitude(m);
#pragma unroll
    for (int c = 0; c < 3; ++c) mw[c] = c == lc[k] ? max(mw[c], finite_bits(m)) : mw[c];
  }
  if (threadIdx.x < 27) {
    mb = finite_bits(b[threadIdx.x]);
    bad |= magnitude(b[threadIdx.x]) >= kInfinity;
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) mw[c] = wave_max(mw[c]);
  mb = wave_max(mb);
  bad = wave_max(bad);
  if ((threadIdx.x & 63) == 0) {
    for (int c = 0; c < 3; ++c) sh[c][threadIdx.x >> 6] = mw[c];
    sh[3][threadIdx.x >> 6] = mb;
    sh[4][threadIdx.x >> 6] = bad;
  }
  __syncthreads();
  int ew[3];
  for (int c = 0; c < 3; ++c) {
    const unsigned m = max(max(sh[c][0], sh[c][1]), max(sh[c][2], sh[c][3]));
    ew[c] = m == 0u ? kNone : min(kTarget - exponent_of(m), 126);
  }
  mb = max(max(sh[3][0], sh[3][1]), max(sh[3][2], sh[3][3]));
  bad = sh[4][0] | sh[4][1] | sh[4][2] | sh[4][3];
  const int nw = (int)(pack_w_bytes(C) / sizeof(f16));
  f16* __restrict__ wp = (f16*)(out + kHeaderBytes);
  float* __restrict__ bp = (float*)(out + kHeaderBytes + pack_w_bytes(C));
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int e = blockIdx.x * 512 + k * kThreads + threadIdx.x;  // nw is a multiple of 512
    const int j = e % 8, lane = (e / 8) % 64, c = (e / 512) % C, kc = (e / (512 * C)) % 2;
    const int part = (e / (1024 * C)) % 2, par = e / (2048 * C);
    const int m = lane & 31;  // row of D: register i of lane half h
    const int p = reg_tap((m >> 2) & 1, 4 * (m >> 3) + (m & 3)), q = slot_tap(par, lane >> 5, kc, j);
    const int es = c == 0 ? ew[0] : c == 1 ? ew[1] : ew[2];
    float v = 0.f;
    if (p >= 0 && q >= 0 && es != kNone) {
      const float w = W[((long)p * C + c) * 27 + q] * pow2(es);
      const f16 hi = (f16)w;
      v = part == 0 ? (float)hi : w - (float)hi;
    }
    wp[e] = (f16)v;
  }
  float* __restrict__ xp = (float*)(out + pack_exact_at(C));
  for (int e = blockIdx.x * kThreads + threadIdx.x; e < (27 * C + 1) * 32; e += gridDim.x * kThreads) {
    const int p = reg_tap((e >> 4) & 1, e & 15), q = e >> 5;
    xp[e] = p < 0 ? 0.f : q == 27 * C ? b[p] : W[((long)p * C + q / 27) * 27 + q % 27];
  }
  if (blockIdx.x != 0) return;
  unsigned small = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int es = lc[k] == 0 ? ew[0] : lc[k] == 1 ? ew[1] : ew[2];
    if (es != kNone) small |= (line[k] << 1) - 1u < least_bits(es);
  }
  small = __syncthreads_or((int)small);
  if (threadIdx.x < 32) {
    const int m = threadIdx.x, p = reg_tap((m >> 2) & 1, 4 * (m >> 3) + (m & 3));
    bp[threadIdx.x] = p >= 0 ? b[p] : 0.f;
  }
  if (threadIdx.x == 0) {
    PackHeader h;
    for (int c = 0; c < 3; ++c) h.w_exp[c] = ew[c];
    h.bias_limit = mb == 0u ? kNone : kOne + kTarget - exponent_of(mb);
    h.finite = bad ? 0 : 1;
    h.exact = bad || small ? 1 : 0;
    *(PackHeader*)out = h;
  }
}

// a + b after lanes 32..63 of a are traded with lanes 0..31 of b: the lower lanes receive
// the sum of a's halves, the upper lanes that of b's.  (Both results pass through an empty
// asm: the ROCm 7.2 compiler otherwise reads the second from the first's register.)
__device__ __forceinline__ float halves_sum(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b),
                                                  false, false);
  unsigned u = r[0], v = r[1];
  asm volatile("" : "+v"(u), "+v"(v));
  return __builtin_bit_cast(float, u) + __builtin_bit_cast(float, v);
}
__device__ __forceinline__ unsigned both_lo(unsigned a, unsigned b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
__device__ __forceinline__ unsigned both_hi(unsigned a, unsigned b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

// PJ: staged rows per plane, halo included
__host__ __device__ constexpr int tile_rows(int FI, int PJ = kPJ) { return (FI + 2) * PJ; }
__host__ __device__ constexpr int tile_cells(int FI, int PJ = kPJ) { return tile_rows(FI, PJ) * kPitch; }

// Position of a tile: the grid's tiles in z, then j, then i order (XCD-contiguous), z rotated
// from row to row of tiles: workgroups go to the shader engines in turn, and the cheap tiles
// (air above the water) have to fall to all of them (256^3, 55 % fluid: 113 -> 105 us).
struct Tile {
  int i0, j0, z0;
};
template <int FI>
__device__ __forceinline__ Tile tile_at(int n2, int n3) {
  const unsigned tz = (unsigned)((n3 + kZ - 1) / kZ), tj = (unsigned)((n2 + kJ - 1) / kJ);
  const unsigned t = xcd_block(blockIdx.x, gridDim.x), u = t / tz;
  return Tile{(int)(u / tj) * FI, (int)(u % tj) * kJ, (int)((t + u) % tz) * kZ};
}

// Raw cells of a staged tile as FP32.  A wave holds rows w, w + 4, ... of every plane, cell
// z0 + lane of each; where PJ is no multiple of 4, its rows start at (w + 2) % 4 in odd planes, so
// that each wave has the last two rows' share in every other plane.  And one z-halo cell of the
// whole tile per thread (rows' cells z0 - 1 and z0 + 64).
template <int FI, int PJ = kPJ>
struct Raw {
  static constexpr int kPlanes = FI + 2, kGroups = PJ / 4, kExtra = PJ % 4 ? kPlanes / 2 : 0;
  static_assert(PJ % 4 == 0 || (PJ % 4 == 2 && kPlanes % 2 == 0), "rows of a tile over four waves");
  static_assert(2 * tile_rows(FI, PJ) <= kThreads, "one halo cell per thread");
  float m[kPlanes][kGroups];
  float x[kExtra ? kExtra : 1];  // row 4 kGroups + w % 2 of plane 2 s + w / 2
  float halo;
  // the wave's first row in planes of parity k
  static __device__ __forceinline__ int row0(int k, int w) { return kExtra ? (w + 2 * (k & 1)) & 3 : w; }
};

// (One resource per plane, whose offsets fit 32 bits, and row offsets shared by the planes of a
// parity: a resource per row took most of the scalar registers and half of the kernel's
// instructions.)
template <int FI, int PJ, typename T>
__device__ __forceinline__ void load_raw(Raw<FI, PJ>& r, const T* __restrict__ src, const Tile& t, int n1, int n2,
                                         int n3, int w, int lane) {
  typedef Raw<FI, PJ> R;
  constexpr unsigned kOut = 0x80000000u;
  const long plane = (long)n2 * n3;
  const int pb = (int)(plane * (int)sizeof(T)), rb = n3 * (int)sizeof(T);
  const unsigned zo = t.z0 + lane < n3 ? (unsigned)(t.z0 + lane) * (unsigned)sizeof(T) : kOut;
  auto load = [&](int k, int row) {
    const int gi = t.i0 + k - 1, gj = t.j0 + row - 1;
    const bool oi = (unsigned)gi < (unsigned)n1, oj = (unsigned)gj < (unsigned)n2;
    return ld_as(rsrc(src + (oi ? gi : 0) * plane, oi ? pb : 0), oj ? zo : kOut, oi && oj ? gj * rb : 0, src);
  };
#pragma unroll
  for (int k = 0; k < R::kPlanes; ++k)
#pragma unroll
    for (int u = 0; u < R::kGroups; ++u) r.m[k][u] = load(k, R::row0(k, w) + 4 * u);
#pragma unroll
  for (int s = 0; s < R::kExtra; ++s) r.x[s] = load(2 * s + (w >> 1), 4 * R::kGroups + (w & 1));
  const int hrow = threadIdx.x >> 1, z = (threadIdx.x & 1) ? t.z0 + kZ : t.z0 - 1;
  const int gi = t.i0 + hrow / PJ - 1, gj = t.j0 + hrow % PJ - 1;
  const bool ok = hrow < tile_rows(FI, PJ) && (unsigned)gi < (unsigned)n1 && (unsigned)gj < (unsigned)n2 &&
                  (unsigned)z < (unsigned)n3;
  r.halo = ok ? (float)src[((long)gi * n2 + gj) * n3 + z] : 0.f;
}

template <int FI, int PJ, typename F>
__device__ __forceinline__ void each_cell(const Raw<FI, PJ>& r, int w, int lane, F&& f) {
  typedef Raw<FI, PJ> R;
#pragma unroll
  for (int k = 0; k < R::kPlanes; ++k)
#pragma unroll
    for (int u = 0; u < R::kGroups; ++u) f(R::row0(k, w) * kPitch + 1 + lane + (k * PJ + 4 * u) * kPitch, r.m[k][u]);
#pragma unroll
  for (int s = 0; s < R::kExtra; ++s)
    f(((w >> 1) * PJ + (w & 1)) * kPitch + 1 + lane + (2 * s * PJ + 4 * R::kGroups) * kPitch, r.x[s]);
  if ((int)(threadIdx.x >> 1) < tile_rows(FI, PJ)) f((threadIdx.x >> 1) * kPitch + (threadIdx.x & 1) * (kZ + 1), r.halo);
}

// Whether three cells in a row of a tile, halo included, hold values below `least` only
// (small_bits), not all 0.  src: as for load_raw.
template <int FI, int PJ, typename T>
__device__ __forceinline__ bool has_small_rows(const Raw<FI, PJ>& r, const T* __restrict__ src, const Tile& t, int n1,
                                               int n2, int n3, unsigned least) {
  typedef Raw<FI, PJ> R;
  bool bad = false;
  auto row = [&](float cell) {
    const float v = fabsf(cell);
    bad |= small_bits(fmaxf(v, fmaxf(wave_from_prev(v), wave_from_next(v)))) < least;
  };
#pragma unroll
  for (int k = 0; k < R::kPlanes; ++k)
#pragma unroll
    for (int u = 0; u < R::kGroups; ++u) row(r.m[k][u]);
#pragma unroll
  for (int s = 0; s < R::kExtra; ++s) row(r.x[s]);
  if (r.halo != 0.f) {  // (then its row is in the grid) with the two cells next to it
    const int hrow = threadIdx.x >> 1, z = (threadIdx.x & 1) ? t.z0 + kZ - 1 : t.z0;
    const T* p = src + ((long)(t.i0 + hrow / PJ - 1) * n2 + t.j0 + hrow % PJ - 1) * n3;
    float v = fmaxf(fabsf(r.halo), fabsf((float)p[z]));
    const int z2 = (threadIdx.x & 1) ? z - 1 : z + 1;
    if (z2 < n3) v = fmaxf(v, fabsf((float)p[z2]));
    bad |= small_bits(v) < least;
  }
  return bad;
}

// The image tile of C channels as two FP16 arrays hi, lo [C][cells], the channels scaled by 2^f,
// or, for exact stencils, as it is, [C][cells] in the same space (T: its type; a BF16 image has
// no lo, it is exact in one FP16 value down to 2^-17).  Ends in a barrier; sh: 4 (C + 2) words of
// LDS; flags: of the wave (uniform), or-ed over the workgroup's; img, t: where raw is from.
template <int C>
struct ImageTile {
  int E, f[C];     // K is scaled by 2^E
  unsigned flags;  // as passed
  bool nonfinite, exact, has_lo;
};
template <typename T, int C, int FI, int PJ>
__device__ __forceinline__ ImageTile<C> stage_image(const Raw<FI, PJ> (&raw)[C], const PackHeader* hd, unsigned flags,
                                                    unsigned exact_flags, int w, int lane, char* im, unsigned* sh,
                                                    const T* __restrict__ img, const Tile& t, int n1, int n2, int n3) {
  constexpr bool LO = sizeof(T) == 4;
  constexpr int kCells = tile_cells(FI, PJ), kS = C + 2;
  f16 *hi = (f16*)im, *lo = hi + C * kCells;
  unsigned mx[C], mn[C], most = 0;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    float m = 0.f;
    mn[c] = ~0u;
    each_cell<FI, PJ>(raw[c], w, lane, [&](int, float v) {
      m = max_nan(m, fabsf(v));
      mn[c] = min(mn[c], small_bits(v));
    });
    mx[c] = magnitude(m);
    most = max(most, mx[c]);
  }
  const bool bad = __builtin_amdgcn_ballot_w64(most >= kInfinity) != 0;
  if (bad) {
    for (int c = 0; c < C; ++c) {
      mx[c] = 0;
      each_cell<FI, PJ>(raw[c], w, lane, [&](int, float v) { mx[c] = max(mx[c], finite_bits(v)); });
    }
  }
#pragma unroll
  for (int c = 0; c < C; ++c) mx[c] = wave_max(mx[c]);
  if (lane == 0) {
#pragma unroll
    for (int c = 0; c < C; ++c) sh[kS * w + c] = mx[c];
    sh[kS * w + C] = (bad ? 1u : 0u) | flags << 1;
  }
  __syncthreads();
  const unsigned all = (unsigned)__builtin_amdgcn_readfirstlane(
      (int)(sh[C] | sh[kS + C] | sh[2 * kS + C] | sh[3 * kS + C]));
  ImageTile<C> it;
  it.nonfinite = (all & 1) != 0;
  it.flags = all >> 1;
  it.E = hd->bias_limit;
  int own[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const unsigned m = max(max(sh[c], sh[kS + c]), max(sh[2 * kS + c], sh[3 * kS + c]));
    own[c] = min(kTarget - exponent_of(m), 126);
    if (m != 0u && hd->w_exp[c] != kNone) it.E = min(it.E, hd->w_exp[c] + own[c]);
  }
  it.E = __builtin_amdgcn_readfirstlane(it.E == kNone ? 0 : it.E);
  bool small = false;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    // (below -126 only where the rows are small, or there is no weight)
    it.f[c] = __builtin_amdgcn_readfirstlane(max(hd->w_exp[c] == kNone ? own[c] : min(it.E - hd->w_exp[c], 126), -126));
    small |= mn[c] < least_bits(it.f[c] + (LO ? 0 : 15));
  }
  it.exact = __builtin_amdgcn_readfirstlane(hd->exact) != 0 || it.nonfinite || (it.flags & exact_flags) != 0;
  it.has_lo = false;
  auto store_raw = [&](const Raw<FI, PJ>& r, int c) {
    each_cell<FI, PJ>(r, w, lane, [&](int e, float v) { ((T*)im)[c * kCells + e] = (T)v; });
  };
  if (it.exact) {
#pragma unroll
    for (int c = 0; c < C; ++c) store_raw(raw[c], c);
    __syncthreads();
    return it;
  }
  unsigned any = 0;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const float s = pow2(it.f[c]);
    each_cell<FI, PJ>(raw[c], w, lane, [&](int e, float v) {
      const float sv = v * s;
      const f16 h = (f16)sv;
      hi[c * kCells + e] = h;
      if (LO) {
        const f16 l = (f16)(sv - (float)h);
        lo[c * kCells + e] = l;
        any |= __builtin_bit_cast(unsigned short, l) & 0x7fffu;
      }
    });
  }
  const bool has = LO && __builtin_amdgcn_ballot_w64(any != 0) != 0, few = __builtin_amdgcn_ballot_w64(small) != 0;
  if (lane == 0) sh[kS * w + C + 1] = (has ? 1u : 0u) | (few ? 2u : 0u);
  __syncthreads();
  const unsigned got = (unsigned)__builtin_amdgcn_readfirstlane(
      (int)(sh[C + 1] | sh[kS + C + 1] | sh[2 * kS + C + 1] | sh[3 * kS + C + 1]));
  it.has_lo = (got & 1) != 0;
  if (got & 2) {  // rare: are small values alone in their rows?
    const long V = (long)n1 * n2 * n3;
    bool rows = false;
#pragma unroll 1
    for (int c = 0; c < C; ++c) {
      Raw<FI, PJ> r;  // (read again: kept, the cells would take registers from everyone)
      load_raw<FI, PJ>(r, img + c * V, t, n1, n2, n3, w, lane);
      int fc = it.f[0];
#pragma unroll
      for (int k = 1; k < C; ++k) fc = c == k ? it.f[k] : fc;
      rows |= has_small_rows<FI, PJ>(r, img + c * V, t, n1, n2, n3, least_bits(fc + (LO ? 0 : 15)));
    }
    it.exact = __syncthreads_or((int)rows) != 0;
    if (it.exact) {
#pragma unroll 1
      for (int c = 0; c < C; ++c) {
        Raw<FI, PJ> r;
        load_raw<FI, PJ>(r, img + c * V, t, n1, n2, n3, w, lane);
        store_raw(r, c);
      }
      __syncthreads();
    }
  }
  return it;
}

// A lane's packed weights, and the first product of one chunk for one z parity.
template <int C>
struct Weights {
  h8 w[2][2][2][C];  // [parity][hi, lo][k half][channel]
  __device__ __forceinline__ void load(const void* pack, int lane) {
    const f16* p = (const f16*)((const char*)pack + kHeaderBytes);
#pragma unroll
    for (int par = 0; par < 2; ++par)
#pragma unroll
      for (int part = 0; part < 2; ++part)
#pragma unroll
        for (int kc = 0; kc < 2; ++kc)
#pragma unroll
          for (int c = 0; c < C; ++c)
            w[par][part][kc][c] = *(const h8*)(p + ((((par * 2 + part) * 2 + kc) * C + c) * 64 + lane) * 8);
  }
  // the bias of the lane's row of D, scaled by 2^(E - kOne): hi and lo on the spare slot of the lower lane
  // half, the rest on that of the upper one
  __device__ __forceinline__ void set_bias(float b, int h) {
    const f16 hi = (f16)b, lo = (f16)(b - (float)hi), rest = (f16)(b - (float)hi - (float)lo);
#pragma unroll
    for (int par = 0; par < 2; ++par) {
      w[par][0][1][0][spare_slot(par)] = h == 0 ? hi : rest;
      w[par][1][1][0][spare_slot(par)] = h == 0 ? lo : (f16)0.f;
    }
  }
};

// byte offsets of the lane's columns' words in a tile of 2-byte cells, at the wave's first chunk
// (row: its staged row less the halo)
struct WordBase {
  unsigned b0[5], b1[5];
  template <int PJ = kPJ>
  __device__ __forceinline__ void init(int h, int n, int row) {
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      const int c = h == 0 ? col_of(0, i) : col_of(1, i);
      b0[i] = (unsigned)((((c / 3) * PJ + c % 3 + row) * kPitch + 2 * n) * 2);
      b1[i] = b0[i] + 4;
      // opaque, so that no two reads are merged into one that needs an address of its own
      asm volatile("" : "+v"(b0[i]), "+v"(b1[i]));
    }
  }
};
// The lane's words of one FP16 array at a chunk as the B operands of the two k halves, per z
// parity; the spare half word (a cell outside the patch) becomes 2^kOne for the bias, or 0.
template <bool ONE>
__device__ __forceinline__ void operands(const f16* arr, const WordBase& wb, int cell, h8 (&b)[2][2]) {
  constexpr unsigned one_hi = ONE ? 0x78000000u : 0u, one_lo = ONE ? 0x7800u : 0u;  // 2^kOne
  const char* p = (const char*)arr + 2 * cell;
  auto word = [&](unsigned off) { return *(const unsigned*)(p + off); };
  const u32x4s e = {word(wb.b0[0]), word(wb.b0[1]), word(wb.b0[2]), word(wb.b0[3])};
  const u32x4s o = {word(wb.b1[0]), word(wb.b1[1]), word(wb.b1[2]), word(wb.b1[3])};
  const unsigned e4 = word(wb.b0[4]), o4 = word(wb.b1[4]);
  b[0][0] = __builtin_bit_cast(h8, e);
  b[0][1] = __builtin_bit_cast(h8, u32x4s{e4, both_lo(o[0], o[1]), both_lo(o[2], o[3]), (o4 & 0xffffu) | one_hi});
  b[1][0] = __builtin_bit_cast(h8, o);
  b[1][1] = __builtin_bit_cast(h8, u32x4s{o4, both_hi(e[0], e[1]), both_hi(e[2], e[3]), (e4 & 0xffff0000u) | one_lo});
}
// scaled K of the lane's columns for both parities, from the tile at `cell`; the products with a
// low part before the others, whose sums they would otherwise be rounded into (FIRST: of all
// channels, whose image words then wait in 16 registers each; else channel by channel), then the
// half with the bias.  Norm-wise error over 24 blocks of random weights, C = 1 and 3, images of
// flags: half by half 9.9e-8 and 1.05e-7, so 9.4e-8 and 9.4e-8; a plan at 256^3 2.20e-7, bias last
// 2.27e-7, bias first 2.08e-7.
template <int C, bool LO, bool FIRST = true>
__device__ __forceinline__ void stencils(const Weights<C>& W, const f16* hi, const f16* lo, int cells,
                                         const WordBase& wb, int cell, f16x (&K)[2]) {
  h8 bh[C][2][2];
  auto high = [&](int c) {
#pragma unroll
    for (int kc = 1; kc >= 0; --kc)
#pragma unroll
      for (int par = 0; par < 2; ++par)
        K[par] = __builtin_amdgcn_mfma_f32_32x32x16_f16(W.w[par][0][kc][c], bh[c][par][kc], K[par], 0, 0, 0);
  };
#pragma unroll
  for (int c = 0; c < C; ++c) {
    h8 bl[2][2];
    if (c == 0) operands<true>(hi, wb, cell, bh[c]);
    else operands<false>(hi + c * cells, wb, cell, bh[c]);
    if (LO) operands<false>(lo + c * cells, wb, cell, bl);
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
#pragma unroll
      for (int par = 0; par < 2; ++par) {
        const f16x in = c == 0 && kc == 0 ? f16x{} : K[par];
        K[par] = __builtin_amdgcn_mfma_f32_32x32x16_f16(W.w[par][1][kc][c], bh[c][par][kc], in, 0, 0, 0);
        if (LO) K[par] = __builtin_amdgcn_mfma_f32_32x32x16_f16(W.w[par][0][kc][c], bl[par][kc], K[par], 0, 0, 0);
      }
    }
    if (!FIRST) high(c);
  }
  if (FIRST) {
#pragma unroll
    for (int c = 0; c < C; ++c) high(c);
  }
}

// The same, not scaled, by FP32 FMAs over the image `at` of a tile cell; cell: that of tap 0 of
// the lane's even voxel.
template <int C, int PJ, typename At>
__device__ __forceinline__ void exact_stencils(const void* pack, int cells, int cell, int h, f16x (&K)[2], At&& at) {
  const float* w = (const float*)((const char*)pack + pack_exact_at(C)) + 16 * h;
#pragma unroll
  for (int i = 0; i < 15; ++i) K[0][i] = K[1][i] = w[27 * C * 32 + i];
  K[0][15] = K[1][15] = 0.f;
#pragma unroll 1
  for (int c = 0; c < C; ++c) {
#pragma unroll 1
    for (int k = 0; k < 9; ++k) {
      const int e = c * cells + cell + (k / 3 * PJ + k % 3) * kPitch;
      const float f[4] = {at(c, e), at(c, e + 1), at(c, e + 2), at(c, e + 3)};
#pragma unroll
      for (int d = 0; d < 3; ++d) {
#pragma unroll
        for (int i = 0; i < 15; ++i) {
          K[0][i] = fmaf(w[i], f[d], K[0][i]);
          K[1][i] = fmaf(w[i], f[d + 1], K[1][i]);
        }
        w += 32;
      }
    }
  }
  // (the upper lanes' fifth column is a dummy, and 0 times an infinity would stay)
#pragma unroll
  for (int i = 12; i < 15; ++i) {
    K[0][i] = h ? 0.f : K[0][i];
    K[1][i] = h ? 0.f : K[1][i];
  }
}

constexpr int kEpiPrev = 1, kEpiMaskA = 2, kEpiMaskB = 4, kEpiDot0 = 8, kEpiDot1 = 16, kEpiRuntime = -1;

// registers for this many waves per SIMD
__host__ __device__ constexpr int split_waves(int C, int BB) { return C == 1 ? (BB == 1 ? 4 : 3) : 2; }

// The apply.  EPI: compile-time epilogue (kEpiRuntime: every operand tested), PL: also write
// the 2x2x2 means of y; BB: right-hand sides per workgroup (K is shared by them).  T: the type of
// x, image and y; a BF16 image is exact in one FP16 value.
template <typename T, int C, int FI, int BB, int EPI, bool PL>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(split_waves(C, BB), 8)))
void sm_split_kernel(SplitArgs a) {
  constexpr int kCells = tile_cells(FI);
  constexpr bool FULL = sizeof(T) == 4;
  __shared__ __attribute__((aligned(16))) float xs[BB][kCells];
  __shared__ __attribute__((aligned(16))) char im[C * kCells * (FULL ? 4 : 2)];
  __shared__ unsigned sh[4 * (C + 2)];
  const f16 *ih = (const f16*)im, *il = ih + C * kCells;
  if (solve_done(a.done)) return;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = lane >> 5, n = lane & 31;
  const Tile t = tile_at<FI>(a.n2, a.n3);
  const long V = (long)a.n1 * a.n2 * a.n3;
  const int b0 = blockIdx.y * BB;

  Raw<FI> rx[BB], ri[C];
#pragma unroll
  for (int c = 0; c < C; ++c) load_raw<FI, kPJ>(ri[c], (const T*)a.img + c * V, t, a.n1, a.n2, a.n3, w, lane);
#pragma unroll
  for (int bb = 0; bb < BB; ++bb)
    if (BB == 1 || b0 + bb < a.B) load_raw<FI, kPJ>(rx[bb], (const T*)a.x + (long)(b0 + bb) * V, t, a.n1, a.n2, a.n3, w, lane);
  const PackHeader* hd = (const PackHeader*)a.pack;
  const float scale = a.in_scale ? (float)(*a.in_scale) : 1.f;
  const float c0 = a.prev ? *a.c0 : 0.f, c1 = a.prev ? *a.c1 : 0.f;

  float xm = 0.f;
#pragma unroll
  for (int bb = 0; bb < BB; ++bb) {
    if (BB > 1 && b0 + bb >= a.B) break;
    each_cell<FI, kPJ>(rx[bb], w, lane, [&](int e, float v) {
      xs[bb][e] = v;
      xm = max_nan(xm, fabsf(v));
    });
  }
  constexpr unsigned kSome = 1, kLarge = 2;  // x is not 0 everywhere; too large for a scaled K
  const unsigned xf = (__builtin_amdgcn_ballot_w64(xm != 0.f) ? kSome : 0u) | (__builtin_amdgcn_ballot_w64(!(xm < kHuge)) ? kLarge : 0u);
  const ImageTile<C> it =
      stage_image<T, C, FI, kPJ>(ri, hd, xf, kLarge, w, lane, im, sh, (const T*)a.img, t, a.n1, a.n2, a.n3);
  Weights<C> W;
  W.load(a.pack, lane);
  W.set_bias(ldexpf(((const float*)((const char*)a.pack + kHeaderBytes + pack_w_bytes(C)))[lane & 31], it.E - kOne), h);
  // x = 0 everywhere: every finite K gives y = 0
  const bool zero = !(it.flags & kSome) && !it.nonfinite && __builtin_amdgcn_readfirstlane(hd->finite);
  const int back = it.exact ? 0 : -it.E;

  WordBase wb;
  wb.init(h, n, w);
  unsigned xb[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) xb[i] = wb.b0[i] * 2;
  const bool dummy = h == 1;  // its fifth column carries no taps
  const int myz = 2 * n + h;
  const bool zok = t.z0 + myz < a.n3;

  constexpr bool RT = EPI == kEpiRuntime;
  constexpr bool LP = RT || (EPI & kEpiPrev), LA = RT || (EPI & kEpiMaskA), LB = RT || (EPI & kEpiMaskB);
  constexpr bool LD0 = RT || (EPI & kEpiDot0), LD1 = RT || (EPI & kEpiDot1);
  const bool has_p = RT ? a.prev != nullptr : LP, has_a = RT ? a.mask_a != nullptr : LA;
  const bool has_b = RT ? a.mask_b != nullptr : LB, has_0 = RT ? a.partials != nullptr : LD0;
  const bool has_1 = RT ? a.dot1 != nullptr : LD1;
  double red[2] = {0.0, 0.0};
  float pp[PL ? FI * 2 : 1];
  const int rows_i = a.n1 - t.i0, rows_j = a.n2 - t.j0;
  const long plane = (long)a.n2 * a.n3, v00 = ((long)t.i0 * a.n2 + t.j0 + w) * a.n3 + t.z0, j4 = 4L * a.n3;
  T* __restrict__ y = (T*)a.y + b0 * V;

  auto chunks = [&](auto mode) {
    constexpr int M = decltype(mode)::value;  // 0: hi alone, 1: hi and lo, 2: exact stencils
#pragma unroll
    for (int q = 0; q < FI * 2; ++q) {
      const int ii = q >> 1, jj = w + 4 * (q & 1);
      if (PL) pp[q] = 0.f;
      if (ii >= rows_i || jj >= rows_j) continue;  // uniform
      const long vr = v00 + ii * plane + (q & 1) * j4;  // uniform; the lane's voxel is vr + myz
      uint8_t ka = 1, kb = 1;
      float pv = 0.f, da = 0.f, db = 0.f;
      if (zok) {
        if (LB && has_b) kb = (a.mask_b + vr)[myz];
        if (LA && has_a) ka = (a.mask_a + vr)[myz];
        if (LP && has_p) pv = (a.prev + vr)[myz];
        if (LD0 && has_0) da = (a.dot0 + vr)[myz];
        if (LD1 && has_1) db = (a.dot1 + vr)[myz];
      }
      constexpr int kHop = kPJ * kPitch;
      const int cell = ii * kHop + 4 * (q & 1) * kPitch;
      float val[BB];
#pragma unroll
      for (int bb = 0; bb < BB; ++bb) val[bb] = 0.f;
      // a chunk that the output mask clears needs no products
      const bool skip = zero || (LB && has_b && __builtin_amdgcn_ballot_w64(zok && kb != 0) == 0);
      if (!skip) {
        f16x K[2];
        if constexpr (M == 2)
          exact_stencils<C, kPJ>(a.pack, kCells, cell + w * kPitch + 2 * n, h, K, [&](int, int e) { return (float)((const T*)im)[e]; });
        else
          stencils<C, M == 1>(W, ih, il, kCells, wb, cell, K);
#pragma unroll
        for (int bb = 0; bb < BB; ++bb) {
          float pe = 0.f, po = 0.f;
          const char* xp = (const char*)xs[bb] + 4 * cell;
#pragma unroll
          for (int i = 0; i < 5; ++i) {
            const float2 u = *(const float2*)(xp + xb[i]), v = *(const float2*)(xp + xb[i] + 8);
            float f[4] = {u.x, u.y, v.x, v.y};
            if (i == 4) {
#pragma unroll
              for (int k = 0; k < 4; ++k) f[k] = dummy ? 0.f : f[k];
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) {
              pe = fmaf(K[0][3 * i + k], f[k], pe);
              po = fmaf(K[1][3 * i + k], f[k + 1], po);
            }
          }
          val[bb] = ldexpf(halves_sum(pe, po), back) * scale;
        }
      }
#pragma unroll
      for (int bb = 0; bb < BB; ++bb) {
        if (BB > 1 && b0 + bb >= a.B) break;
        float v = val[bb];
        if (LA && has_a && ka == 0) v = 0.f;
        if (LP && has_p) v = c0 * pv + c1 * v;
        if (LB && has_b && kb == 0) v = 0.f;
        if (zok) (y + bb * V + vr)[myz] = (T)v;
        if (PL) pp[q] = halves_sum(v, v);
        if (LD0 && has_0) {
          red[0] += (double)v * (double)da;
          if (LD1 && has_1) red[1] += (double)v * (double)db;
          asm volatile("" : "+v"(red[0]), "+v"(red[1]));  // see sm_fused_kernel
        }
      }
    }
  };
  if (it.exact) chunks(std::integral_constant<int, 2>());
  else if (FULL && it.has_lo && !zero) chunks(std::integral_constant<int, FULL ? 1 : 0>());
  else chunks(std::integral_constant<int, 0>());
  if (LD0 && has_0) block_partials<2>(red, a.partials);
  if constexpr (PL) {
    // the means of the stored output in avgpool2_kernel's order (z pair, then rows 2J, 2J + 1
    // of plane 2I, then of 2I + 1); the rows of a mean belong to two waves, so the pair sums
    // meet in LDS (in the x tile's space)
    __syncthreads();
    float* P = &xs[0][0];  // [FI][8 rows][32]
    static_assert(FI * 8 * 32 <= kCells, "pair sums fit the x tile");
    if (h == 0) {
#pragma unroll
      for (int q = 0; q < FI * 2; ++q) P[((q >> 1) * 8 + w + 4 * (q & 1)) * 32 + n] = pp[q];
    }
    __syncthreads();
    const int c1n = a.n1 >> 1, c2n = a.n2 >> 1, c3n = a.n3 >> 1;
    for (int e = threadIdx.x; e < (FI / 2) * 4 * 32; e += kThreads) {
      const int kc = e & 31, J = (e >> 5) & 3, I = e >> 7;
      const int gi = t.i0 / 2 + I, gj = t.j0 / 2 + J, gk = t.z0 / 2 + kc;
      const float* p0 = P + (2 * I * 8 + 2 * J) * 32 + kc;
      const float sum = ((p0[0] + p0[32]) + p0[8 * 32]) + p0[8 * 32 + 32];
      if (gi < c1n && gj < c2n && gk < c3n) a.pool_out[((long)gi * c2n + gj) * c3n + gk] = sum * 0.125f;
    }
  }
}

// Host side -----------------------------------------------------------------------------

// Planes per tile: deeper tiles stage fewer halo cells per voxel, but a grid needs enough
// workgroups to fill the chip.
constexpr unsigned kMinBlocks = 1024;
inline unsigned blocks_at(int FI, int n1, int n2, int n3) {
  return (unsigned)((n1 + FI - 1) / FI) * (unsigned)((n2 + kJ - 1) / kJ) * (unsigned)((n3 + kZ - 1) / kZ);
}
inline int planes(int n1, int n2, int n3) { return blocks_at(4, n1, n2, n3) >= kMinBlocks ? 4 : 2; }

template <int C, int BB, int EPI, bool PL, typename T = float>
void launch(const SplitArgs& a, hipStream_t st) {
  const int fi = planes(a.n1, a.n2, a.n3);
  const dim3 g(blocks_at(fi, a.n1, a.n2, a.n3), (unsigned)((a.B + BB - 1) / BB));
  if (fi == 4) sm_split_kernel<T, C, 4, BB, EPI, PL><<<g, kThreads, 0, st>>>(a);
  else sm_split_kernel<T, C, 2, BB, EPI, PL><<<g, kThreads, 0, st>>>(a);
}

// Compile-time epilogues for the launches of a preconditioner application and of block
// forwards; the rest (the model's mask) test their operands.
template <int C>
void launch_epi(const SplitArgs& a, hipStream_t st) {
  const int epi = (a.prev ? kEpiPrev : 0) | (a.mask_a ? kEpiMaskA : 0) | (a.mask_b ? kEpiMaskB : 0) |
                  (a.partials ? kEpiDot0 : 0) | (a.partials && a.dot1 ? kEpiDot1 : 0);
  if (a.is_bf16) return a.B > 1 ? launch<C, 2, 0, false, bf16>(a, st) : launch<C, 1, 0, false, bf16>(a, st);
  if (epi == 0 && a.pool_out) return launch<C, 1, 0, true>(a, st);
  if (epi == 0 && a.B > 1) return launch<C, 2, 0, false>(a, st);
  if (epi == 0) return launch<C, 1, 0, false>(a, st);
  if (epi == kEpiPrev) return launch<C, 1, kEpiPrev, false>(a, st);
  if (epi == (kEpiPrev | kEpiMaskB | kEpiDot0)) return launch<C, 1, kEpiPrev | kEpiMaskB | kEpiDot0, false>(a, st);
  if (epi == (kEpiPrev | kEpiMaskB | kEpiDot0 | kEpiDot1))
    return launch<C, 1, kEpiPrev | kEpiMaskB | kEpiDot0 | kEpiDot1, false>(a, st);
  launch<C, 1, kEpiRuntime, false>(a, st);
}

}  // namespace split

size_t split_pack_bytes(int C) { return split::pack_bytes(C); }

bool split_eligible(int C, int n1, int n2, int n3) {
  // a plane is addressed with 32-bit buffer offsets
  return C >= 1 && C <= 3 && n1 >= 1 && n2 >= 1 && n3 >= 1 && (long)n2 * n3 * 4 < (1L << 31);
}

unsigned split_blocks(int C, int n1, int n2, int n3) {
  return split::blocks_at(split::planes(n1, n2, n3), n1, n2, n3);
}

int launch_split_pack(const void* W, const void* b, int C, void* pack, hipStream_t st) {
  MLPCG_REQUIRE(C >= 1 && C <= 3, "split_pack: C must be 1, 2 or 3 (got %d)", C);
  split::split_pack_kernel<<<8 * C, kThreads, 0, st>>>((const float*)W, (const float*)b, C, (char*)pack);
  return check_launch("split_pack");
}

// Error against 64 bits (norm-wise, the modules' weights, random and flag images): C = 1
// 1.08e-7 and 0.95e-7 where the FP32 chain of the stored stencils has 1.18e-7 and 1.10e-7;
// C = 3 1.25e-7 and 0.99e-7 against 1.77e-7 and 1.38e-7.
// Time of a block forward (packing included), stored stencils -> now: 256^3 C = 1 843 ->
// 100 us, C = 3 1483 -> 244 us; 128^3 C = 1 90 -> 22 us, two right-hand sides 97 -> 30 us,
// C = 3 185 -> 39 us; 97 x 75 x 131 C = 3, two right-hand sides 103 -> 38 us; at 32^3 both
// take the 19 us of two launches.
int launch_sm_split(int C, const SplitArgs& a, hipStream_t st) {
  MLPCG_REQUIRE(split_eligible(C, a.n1, a.n2, a.n3), "sm_split: grid (%d,%d,%d) / C=%d not supported", a.n1, a.n2,
                a.n3, C);
  const bool epi = a.prev || a.mask_a || a.mask_b || a.partials;
  MLPCG_REQUIRE(a.B >= 1 && (a.B == 1 || (!epi && !a.pool_out)), "sm_split: epilogues need B = 1");
  MLPCG_REQUIRE(!a.is_bf16 || (!epi && !a.pool_out), "sm_split: BF16 blocks have no epilogue");
  MLPCG_REQUIRE((!a.partials || a.dot0) && (!a.dot1 || a.dot0), "sm_split: dot sums need dot0");
  MLPCG_REQUIRE(!a.pool_out || (!epi && a.n1 % 2 == 0 && a.n2 % 2 == 0 && a.n3 % 2 == 0),
                "sm_split: the pooled output needs an even grid and no epilogue operands");
  // a launch takes 65535 workgroups of two right-hand sides at most
  constexpr int kMost = 2 * 65535;
  const size_t V = (size_t)a.n1 * a.n2 * a.n3, es = a.is_bf16 ? 2 : 4;
  for (int b = 0; b < a.B; b += kMost) {
    SplitArgs p = a;
    p.x = (const float*)((const char*)a.x + (size_t)b * V * es);
    p.y = (float*)((char*)a.y + (size_t)b * V * es);
    p.B = a.B - b < kMost ? a.B - b : kMost;
    if (C == 1) split::launch_epi<1>(p, st);
    else if (C == 2) split::launch_epi<2>(p, st);
    else split::launch_epi<3>(p, st);
  }
  return check_launch("sm_split");
}

}  // namespace mlpcg
