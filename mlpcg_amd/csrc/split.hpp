// FP32 SM block on the matrix cores, by FP16 operands split in two.
//
//   y[b, v] = sum_p K_p(v) x[b, v + d_p],   K_p(v) = b_p + sum_{c,s} W[p,c,s] img[c, v + d_s]
//
// (sm_block_3d_kernel.cu:46-70), all in FP32.  K is neither stored nor streamed (108 of the
// 116 bytes per voxel of the stored-stencil apply): it is recomputed from the image tile in
// LDS.  W and the image are scaled by powers of two and split as v = hi + lo into two FP16
// values each, which keeps 22 bits and more, and
//   W . img = W_hi img_hi + W_lo img_hi + W_hi img_lo          (FP16 products, FP32 sums)
// on v_mfma_f32_32x32x16_f16.  The dropped W_lo img_lo is below 2^-22 of its term, the matrix
// cores round once where an FP32 chain rounds 28 times; measured against 64 bits the block's
// error is below that of the FP32 chain (see launch_sm_split).  K meets x in FP32 FMAs.
//
// Scaling.  A workgroup takes the largest finite |img| of its tile and scales it into
// [2^4, 2^5) (exact: a power of two), W likewise over the whole weight when it is packed, so
// images and weights of any magnitude keep their bits: what falls below FP16's denormal
// 2^-24 is below 2^-28 of the largest value.  The bias, scaled by both factors, joins as
// three FP16 parts (33 bits) on spare K slots whose image value is 1 (as an accumulator it
// took 16 registers and a wave per SIMD); where it is large against W img it limits the
// image's factor (the bits lost are far below the bias's own).  y is scaled back once.
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
constexpr int kTarget = 4;      // largest |W| and |img| are scaled into [2^4, 2^5)
constexpr int kBiasTarget = 8;  // and the largest scaled bias stays below 2^9


// column i (0..4) of lane half h; the fifth of the upper half is a dummy (zero weights).  The
// first three are a plane's (d1 = -1, +1), which the input gradient (igrad.hpp) relies on.
__host__ __device__ constexpr int col_of(int h, int i) { return h == 0 ? i : (i < 3 ? 6 + i : i == 3 ? 5 : 8); }
__host__ __device__ constexpr bool col_real(int h, int i) { return h == 0 || i < 4; }

struct PackHeader {
  float inv_scale;  // 1 / (the weights' factor)
  int img_limit;    // largest exponent of the image's factor (from the bias)
  int finite;       // no weight or bias is infinite or NaN
  int pad;
};
// header, then W [parity][hi, lo][k half][channel][lane][8] (FP16), then the scaled bias of
// the 32 rows of D (FP32)
constexpr size_t kHeaderBytes = 64;
constexpr size_t pack_w_bytes(int C) { return (size_t)2 * 2 * 2 * C * 64 * 8 * sizeof(f16); }
constexpr size_t pack_bytes(int C) { return kHeaderBytes + pack_w_bytes(C) + 32 * sizeof(float); }

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
  __shared__ unsigned sh[3][4];
  unsigned mw = 0, mb = 0, bad = 0;
#pragma unroll
  for (int k = 0; k < 9; ++k) {  // C <= 3; clamped, so that all loads are in flight together
    const float v = W[min(k * kThreads + (int)threadIdx.x, 27 * 27 * C - 1)];
    const unsigned u = finite_bits(v);
    mw = mw > u ? mw : u;
    bad |= (__float_as_uint(v) & 0x7f800000u) == 0x7f800000u;
  }
  if (threadIdx.x < 27) {
    mb = finite_bits(b[threadIdx.x]);
    bad |= (__float_as_uint(b[threadIdx.x]) & 0x7f800000u) == 0x7f800000u;
  }
  mw = wave_max(mw);
  mb = wave_max(mb);
  bad = wave_max(bad);
  if ((threadIdx.x & 63) == 0) {
    sh[0][threadIdx.x >> 6] = mw;
    sh[1][threadIdx.x >> 6] = mb;
    sh[2][threadIdx.x >> 6] = bad;
  }
  __syncthreads();
  for (int k = 0; k < 4; ++k) {
    mw = mw > sh[0][k] ? mw : sh[0][k];
    mb = mb > sh[1][k] ? mb : sh[1][k];
    bad |= sh[2][k];
  }
  const int ew = min(kTarget - exponent_of(mw), 100);
  const float s = pow2(ew);
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
    float v = 0.f;
    if (p >= 0 && q >= 0) {
      const float w = W[((long)p * C + c) * 27 + q] * s;
      const f16 hi = (f16)w;
      v = part == 0 ? (float)hi : w - (float)hi;
    }
    wp[e] = (f16)v;
  }
  if (blockIdx.x == 0 && threadIdx.x < 32) {
    const int m = threadIdx.x, p = reg_tap((m >> 2) & 1, 4 * (m >> 3) + (m & 3));
    bp[threadIdx.x] = p >= 0 ? b[p] * s : 0.f;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    PackHeader h;
    h.inv_scale = pow2(-ew);
    h.img_limit = mb == 0u ? 126 : kBiasTarget - (exponent_of(mb) + ew);
    h.finite = bad ? 0 : 1;
    h.pad = 0;
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

// Raw cells of a staged tile as FP32: rows w, w + 4, ... of the wave, cell z0 + lane of each,
// and one z-halo cell of the whole tile per thread (rows' cells z0 - 1 and z0 + 64).
template <int FI, int PJ = kPJ>
struct Raw {
  static constexpr int kRows = (tile_rows(FI, PJ) + 3) / 4;
  static_assert(2 * tile_rows(FI, PJ) <= kThreads, "one halo cell per thread");
  float m[kRows];
  float halo;
};

template <int FI, int PJ, typename T>
__device__ __forceinline__ void load_raw(Raw<FI, PJ>& r, const T* __restrict__ src, const Tile& t, int n1, int n2,
                                         int n3, int w, int lane) {
  const long plane = (long)n2 * n3;
  const int pb = (int)(plane * (int)sizeof(T)), rb = n3 * (int)sizeof(T);
  const unsigned zo = t.z0 + lane < n3 ? (unsigned)(t.z0 + lane) * (unsigned)sizeof(T) : 0x80000000u;
#pragma unroll
  for (int k = 0; k < Raw<FI, PJ>::kRows; ++k) {
    const int row = w + 4 * k;
    const int gi = t.i0 + row / PJ - 1, gj = t.j0 + row % PJ - 1;
    const bool ok = row < tile_rows(FI, PJ) && (unsigned)gi < (unsigned)n1 && (unsigned)gj < (unsigned)n2;
    r.m[k] = ld_as(rsrc(src + (ok ? gi : 0) * plane, ok ? pb : 0), zo, (ok ? gj : 0) * rb, src);
  }
  const int hrow = threadIdx.x >> 1, z = (threadIdx.x & 1) ? t.z0 + kZ : t.z0 - 1;
  const int gi = t.i0 + hrow / PJ - 1, gj = t.j0 + hrow % PJ - 1;
  const bool ok = hrow < tile_rows(FI, PJ) && (unsigned)gi < (unsigned)n1 && (unsigned)gj < (unsigned)n2 &&
                  (unsigned)z < (unsigned)n3;
  r.halo = ok ? (float)src[((long)gi * n2 + gj) * n3 + z] : 0.f;
}

template <int FI, int PJ, typename F>
__device__ __forceinline__ void each_cell(const Raw<FI, PJ>& r, int w, int lane, F&& f) {
#pragma unroll
  for (int k = 0; k < Raw<FI, PJ>::kRows; ++k)
    if (w + 4 * k < tile_rows(FI, PJ)) f((w + 4 * k) * kPitch + 1 + lane, r.m[k]);
  if ((int)(threadIdx.x >> 1) < tile_rows(FI, PJ)) f((threadIdx.x >> 1) * kPitch + (threadIdx.x & 1) * (kZ + 1), r.halo);
}

// The image tile of C channels as two FP16 arrays hi, lo [C][cells].  Returns (uniform) the
// exponent of the tile's factor; flags: any non-finite cell, any nonzero lo (LO = false: the
// image is of a type that hi holds, lo is left out).  Ends in a barrier; sh: 8 words of LDS.
struct ImageTile {
  int exp;
  bool nonfinite, has_lo;
};
template <int C, int FI, int PJ = kPJ, bool LO = true>
__device__ __forceinline__ ImageTile stage_image(const Raw<FI, PJ> (&raw)[C], int limit, int w, int lane, f16* hi, f16* lo,
                                                 unsigned* sh) {
  unsigned m = 0, bad = 0;
#pragma unroll
  for (int c = 0; c < C; ++c)
    each_cell<FI, PJ>(raw[c], w, lane, [&](int, float v) {
      const unsigned u = __float_as_uint(v) & 0x7fffffffu;
      const bool fin = u < 0x7f800000u;
      m = max(m, fin ? u : 0u);
      bad |= fin ? 0u : 1u;
    });
  m = wave_max(m);
  bad = __builtin_amdgcn_ballot_w64(bad != 0) != 0;
  if (lane == 0) {
    sh[w] = m;
    sh[4 + w] = bad;
  }
  __syncthreads();
  m = max(max(sh[0], sh[1]), max(sh[2], sh[3]));
  bad = sh[4] | sh[5] | sh[6] | sh[7];
  ImageTile it;
  it.exp = __builtin_amdgcn_readfirstlane(max(-126, min(min(kTarget - exponent_of(m), limit), 126)));
  it.nonfinite = __builtin_amdgcn_readfirstlane((int)bad) != 0;
  const float s = pow2(it.exp);
  unsigned any = 0;
#pragma unroll
  for (int c = 0; c < C; ++c)
    each_cell<FI, PJ>(raw[c], w, lane, [&](int e, float v) {
      const float sv = v * s;
      const f16 h = (f16)sv;
      hi[c * tile_cells(FI, PJ) + e] = h;
      if (LO) {
        const f16 l = (f16)(sv - (float)h);
        lo[c * tile_cells(FI, PJ) + e] = l;
        any |= __builtin_bit_cast(unsigned short, l) & 0x7fffu;
      }
    });
  if (!LO) {
    it.has_lo = false;
    __syncthreads();
    return it;
  }
  any = __builtin_amdgcn_ballot_w64(any != 0) != 0;
  __syncthreads();  // the flags above were read by everyone
  if (lane == 0) sh[w] = any;
  __syncthreads();
  it.has_lo = __builtin_amdgcn_readfirstlane((int)(sh[0] | sh[1] | sh[2] | sh[3])) != 0;
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
  // the bias of the lane's row of D, scaled: hi and lo on the spare slot of the lower lane
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
// parity; the spare half word (a cell outside the patch) becomes 1 for the bias, or 0.
template <bool ONE>
__device__ __forceinline__ void operands(const f16* arr, const WordBase& wb, int cell, h8 (&b)[2][2]) {
  constexpr unsigned one_hi = ONE ? 0x3c000000u : 0u, one_lo = ONE ? 0x3c00u : 0u;
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
// scaled K of the lane's columns for both parities, from the tile at `cell`
template <int C, bool LO>
__device__ __forceinline__ void stencils(const Weights<C>& W, const f16* hi, const f16* lo, int cells,
                                         const WordBase& wb, int cell, f16x (&K)[2]) {
#pragma unroll
  for (int c = 0; c < C; ++c) {
    h8 bh[2][2], bl[2][2];
    if (c == 0) operands<true>(hi, wb, cell, bh);
    else operands<false>(hi + c * cells, wb, cell, bh);
    if (LO) operands<false>(lo + c * cells, wb, cell, bl);
#pragma unroll
    for (int par = 0; par < 2; ++par) {
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        const f16x in = c == 0 && kc == 0 ? f16x{} : K[par];
        K[par] = __builtin_amdgcn_mfma_f32_32x32x16_f16(W.w[par][1][kc][c], bh[par][kc], in, 0, 0, 0);
        if (LO) K[par] = __builtin_amdgcn_mfma_f32_32x32x16_f16(W.w[par][0][kc][c], bl[par][kc], K[par], 0, 0, 0);
        K[par] = __builtin_amdgcn_mfma_f32_32x32x16_f16(W.w[par][0][kc][c], bh[par][kc], K[par], 0, 0, 0);
      }
    }
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
  __shared__ __attribute__((aligned(16))) f16 ih[C * kCells], il[FULL ? C * kCells : 8];
  __shared__ unsigned sh[12];
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

  unsigned xany = 0;
#pragma unroll
  for (int bb = 0; bb < BB; ++bb) {
    if (BB > 1 && b0 + bb >= a.B) break;
    each_cell<FI, kPJ>(rx[bb], w, lane, [&](int e, float v) {
      xs[bb][e] = v;
      xany |= __float_as_uint(v) & 0x7fffffffu;
    });
  }
  xany = __builtin_amdgcn_ballot_w64(xany != 0) != 0;
  if (lane == 0) sh[8 + w] = xany;
  const ImageTile it = stage_image<C, FI, kPJ, FULL>(ri, hd->img_limit, w, lane, ih, il, sh);
  Weights<C> W;
  W.load(a.pack, lane);
  W.set_bias(((const float*)((const char*)a.pack + kHeaderBytes + pack_w_bytes(C)))[lane & 31] * pow2(it.exp), h);
  // x = 0 everywhere: every finite K gives y = 0
  const bool zero = !__builtin_amdgcn_readfirstlane((int)(sh[8] | sh[9] | sh[10] | sh[11])) && !it.nonfinite &&
                    __builtin_amdgcn_readfirstlane(hd->finite);
  const float inv_i = pow2(-it.exp), inv_w = hd->inv_scale * scale;

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

  auto chunks = [&](auto lo_c) {
    constexpr bool LO = decltype(lo_c)::value;
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
        stencils<C, LO>(W, ih, il, kCells, wb, cell, K);
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
          val[bb] = halves_sum(pe, po) * inv_i * inv_w;
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
  if constexpr (FULL) {
    if (it.has_lo && !zero) chunks(std::true_type());
    else chunks(std::false_type());
  } else {
    chunks(std::false_type());
  }
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
// 1.06e-7 and 0.97e-7 where the FP32 chain of the stored stencils has 1.17e-7 and 1.07e-7;
// C = 3 1.56e-7 and 1.11e-7 against 1.89e-7 and 1.38e-7.
// Time of a block forward (packing included), stored stencils -> now: 256^3 C = 1 843 ->
// 111 us, C = 3 1483 -> 258 us; 128^3 C = 1 90 -> 25 us, two right-hand sides 97 -> 34 us,
// C = 3 185 -> 46 us; 97 x 75 x 131 C = 3, two right-hand sides 103 -> 44 us; at 32^3 both
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
