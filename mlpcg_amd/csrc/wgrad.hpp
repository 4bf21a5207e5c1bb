// Weight gradient of the SM block on the matrix cores, for FP32, BF16 and FP16 data:
//   D[p][q] = sum_v G_p(v) P_q(v),  G_p(v) = sum_b a[b,v] c[b,v+d_p]   (sm_block_3d_kernel.cu:121-229)
// with P_q the 27 C image taps and a column of ones (the bias gradient), a 27 x (27C + 1)
// product over all voxels: gW[p][q] = D[p][q], gb[p] = D[p][27C].
//
// a, c and the image are scaled by powers of two and G, formed in FP32, and P are split into
// two FP16 values each (see split_common.hpp); D = G_hi P_hi + G_lo P_hi + G_hi P_lo on
// v_mfma_f32_32x32x16_f16.  For BF16 data G is exact in its two parts and P in one, so every
// product is exact; tiles whose image has no low part leave the third product out.  The
// products with a low part have accumulators of their own: fewer roundings of the large sums
// (and the matrix cores cut, not round, what is far below their largest addend: adding all
// three to fresh accumulators per row doubled the error).
//
// The factors of a and c (per right-hand side) and of each image channel come from the tile's
// own largest finite magnitudes, and a tile's products are added, scaled back, to FP32 sums
// kept beside its accumulators: no tile's factor reaches another's, whether that is empty or
// its values are far larger.  FP16's smallest step is then 2^-39 of the largest |a| |c| and of
// the largest |image| of a tile.  Where no product of the tile's centre taps comes within 2^-16 of
// the former, all products are looked at and the largest sets the scale of G.  (What is 2^-39
// below a tile's largest G is lost: where x falls off into the air by such factors, the image is
// 0, and the sums' errors stay below the FP32 products'.)  Tiles with three
// image cells in a row that are all 2^-16 and more below the latter, with infinities or with NaN
// are summed in FP32 on the VALU, over the cells and taps inside the grid alone (some 10 times
// slower, for a kind of tile that is rare).  They wait until the workgroup's others are done:
// among them, that code's registers and instructions cost every tile 5 %.
//
// Tile: 4 planes x 8 rows x 64 z; x and the image with a one-cell halo in LDS, any extents.
// A wave takes rows of 64 voxels, 16 voxels per product: lane (h, m) = (lane / 32, lane % 32)
// holds G of tap m and P of column m at voxels 16 s + 8 h + j, j < 8.  The x row and plane
// pitches (67 and 681 words: 3 and 9 mod 32) put the 27 taps of a half-wave's read on 27
// different banks; the image's (34 and 358 words) do the same for its words.  a reaches the
// lanes by a DPP row broadcast inside the multiply (8 LDS reads per product less).  An image tap
// with d3 = +-1 is five words shifted by half a word, so no shifted copies are kept.
//
// Bound by VALU (3 instructions per G: product, difference, two conversions of pairs) and
// LDS reads, about equally, then by the staging of the tiles (a third of the time), all above
// the matrix products.  Before (FP32 matrix products gathered from global memory or staged
// rows, C = 3 on the VALU) -> now: 128^3 FP32 C = 1 88 -> 30 us, two right-hand sides 238 ->
// 44 us, C = 3 576 -> 75 us; 256^3 C = 1 712 -> 190 us.  Errors against 64 bits (norm-wise):
// 0.8 to 1.9e-7 where the FP32 products had 0.8 to 5.2e-7.
#pragma once

#include "kernels.hpp"
#include "split_common.hpp"

namespace mlpcg {
namespace wgrad {

using namespace split;

constexpr int kI = 4, kJ = 8, kZ = 64, kPJ = kJ + 2, kRows = (kI + 2) * kPJ;
constexpr int kXRow = 67, kXPlane = 681;      // x pitches (words); cell z0 - 1 + e at e
constexpr int kIRow = 68, kIPlane = 716;      // image pitches (half words); cell z0 - 1 + e at 1 + e
constexpr int kXCells = (kI + 2) * kXPlane, kICells = (kI + 2) * kIPlane;
static_assert(kXRow % 32 == 3 && kXPlane % 32 == 9 && (kIRow / 2) % 32 == 2 && (kIPlane / 2) % 32 == 6, "banks");
static_assert(kXPlane >= kPJ * kXRow && kIPlane >= kPJ * kIRow, "planes do not overlap");
constexpr int kTargetG = 6, kTargetP = 14;  // |a|, |c| into [2^6, 2^7), |image| into [2^14, 2^15)
constexpr int kQueue = 32;                 // tiles that wait for their FP32 products
constexpr int kOnes = 40;                  // words of FP16 ones, and of zeros, for the bias column
constexpr int kRw = 3;                     // staged rows per wave and plane: j = w, w + 4, w + 8 of 10
static_assert(2 * kRows <= kThreads, "staging");

// FP32 cells of a tile as loaded: cell z0 + lane of the wave's rows, and one of the cells
// z0 - 1, z0 + 64 of all rows
struct Raw {
  float m[kI + 2][kRw];
  float halo;
};

struct Pos {
  int i0, j0, z0;
};

// (a tensor has fewer than 2^31 bytes, so one resource with 32-bit offsets serves all of its rows;
// a base for each row or plane filled the scalar registers and beyond)
constexpr unsigned kOut = 0x80000000u;
template <typename T>
__device__ __forceinline__ void load_tile(Raw& r, const T* __restrict__ src, const Pos& t, int n1, int n2, int n3,
                                          int w, int lane) {
  const int rb = n3 * (int)sizeof(T), pb = n2 * rb;
  const unsigned zo = t.z0 + lane < n3 ? (unsigned)(t.z0 + lane) * (unsigned)sizeof(T) : kOut;
  int so[kRw];
  unsigned vo[kRw];  // kOut in rows outside the grid
#pragma unroll
  for (int u = 0; u < kRw; ++u) {
    const int gj = t.j0 + w + 4 * u - 1;
    const bool ok = (unsigned)gj < (unsigned)n2 && w + 4 * u < kPJ;
    so[u] = ok ? gj * rb : 0;
    vo[u] = ok ? zo : kOut;
  }
#pragma unroll
  for (int k = 0; k < kI + 2; ++k) {
    const int gi = t.i0 + k - 1;
    const bool ok = (unsigned)gi < (unsigned)n1;
    const auto res = rsrc(src, ok ? n1 * pb : 0);
#pragma unroll
    for (int u = 0; u < kRw; ++u) r.m[k][u] = ld_as(res, vo[u], ok ? gi * pb + so[u] : 0, src);
  }
  const int hrow = threadIdx.x >> 1, z = (threadIdx.x & 1) ? t.z0 + kZ : t.z0 - 1;
  const int gi = t.i0 + hrow / kPJ - 1, gj = t.j0 + hrow % kPJ - 1;
  const bool ok = hrow < kRows && (unsigned)gi < (unsigned)n1 && (unsigned)gj < (unsigned)n2 &&
                  (unsigned)z < (unsigned)n3;
  r.halo = ok ? (float)src[((long)gi * n2 + gj) * n3 + z] : 0.f;
}
// f(plane, row, e, value) for the thread's cells (rows of the third group exist for two waves)
template <typename F>
__device__ __forceinline__ void each(const Raw& r, int w, int lane, F&& f) {
#pragma unroll
  for (int u = 0; u < kRw; ++u) {
    if (w + 4 * u >= kPJ) continue;
#pragma unroll
    for (int k = 0; k < kI + 2; ++k) f(k, w + 4 * u, 1 + lane, r.m[k][u]);
  }
  const int hrow = threadIdx.x >> 1;
  if (hrow < kRows) f(hrow / kPJ, hrow % kPJ, (int)(threadIdx.x & 1) * (kZ + 1), r.halo);
}
// largest magnitude (bits; kInfinity or more with an infinite or NaN cell)
__device__ __forceinline__ unsigned max_of(const Raw& r) {
  float m = fabsf(r.halo);
#pragma unroll
  for (int k = 0; k < kI + 2; ++k)
#pragma unroll
    for (int u = 0; u < kRw; ++u) m = max_nan(m, fabsf(r.m[k][u]));
  return magnitude(m);
}
// smallest magnitude that is not 0 (small_bits)
__device__ __forceinline__ unsigned min_of(const Raw& r) {
  unsigned m = small_bits(r.halo);
#pragma unroll
  for (int k = 0; k < kI + 2; ++k)
#pragma unroll
    for (int u = 0; u < kRw; ++u) m = min(m, small_bits(r.m[k][u]));
  return m;
}
// the same of the finite cells alone
__device__ __forceinline__ unsigned finite_max_of(const Raw& r) {
  unsigned m = finite_bits(r.halo);
#pragma unroll
  for (int k = 0; k < kI + 2; ++k)
#pragma unroll
    for (int u = 0; u < kRw; ++u) m = max(m, finite_bits(r.m[k][u]));
  return m;
}
__device__ __forceinline__ int scale_exp(unsigned bits, int target) {
  return max(-126, min(target - exponent_of(bits), 126));
}
// Whether three cells in a row of a tile, halo included, hold values below `least` only
// (small_bits), not all 0.  If not, sums over a patch are as good as if the smaller values were
// held like `least`.  src: as for load_tile.
template <typename T>
__device__ __forceinline__ bool has_small_rows(const Raw& r, const T* __restrict__ src, const Pos& t, int n1, int n2,
                                               int n3, unsigned least) {
  bool bad = false;
#pragma unroll
  for (int k = 0; k < kI + 2; ++k)
#pragma unroll
    for (int u = 0; u < kRw; ++u) {
      const float v = fabsf(r.m[k][u]);
      bad |= small_bits(fmaxf(v, fmaxf(wave_from_prev(v), wave_from_next(v)))) < least;
    }
  if (r.halo != 0.f) {  // (then its row is in the grid) with the two cells next to it
    const int hrow = threadIdx.x >> 1, z = (threadIdx.x & 1) ? t.z0 + kZ - 1 : t.z0;
    const T* p = src + ((long)(t.i0 + hrow / kPJ - 1) * n2 + t.j0 + hrow % kPJ - 1) * n3;
    float v = fmaxf(fabsf(r.halo), fabsf((float)p[z]));
    const int z2 = (threadIdx.x & 1) ? z - 1 : z + 1;
    if (z2 < n3) v = fmaxf(v, fabsf((float)p[z2]));
    bad |= small_bits(v) < least;
  }
  return bad;
}
// lane I of a row of 16 to the whole row
template <int I>
__device__ __forceinline__ float row_bcast(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150 + I, 0xf, 0xf, true));
}
// FP16 parts of two values: hi rounded, lo = v - hi rounded.  The differences are written out
// (a mixed-precision FMA each): left to the ROCm 7.2 compiler, hi is rounded from the exact
// product behind v in one use and from its FP32 value in another, and no longer fits its lo.
typedef f16 h2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void split_pair(float v0, float v1, unsigned& hi, unsigned& lo) {
  float d0, d1;
  asm("" : "+v"(v0), "+v"(v1));
  hi = __builtin_bit_cast(unsigned, h2{(f16)v0, (f16)v1});
  asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[0,0,1]" : "=v"(d0) : "v"(v0), "v"(hi));
  asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(d1) : "v"(v1), "v"(hi));
  lo = __builtin_bit_cast(unsigned, h2{(f16)d0, (f16)d1});
}

// G[j] = (ACC: G[j] +) g of voxel j times x[j].  (Contracted into the difference v - hi, the
// product could not take its broadcast as a DPP operand.)
template <bool ACC>
__device__ __forceinline__ void products(float g, const float (&x)[8], float (&G)[8]) {
#pragma clang fp contract(off)
  const float gb[8] = {row_bcast<0>(g), row_bcast<1>(g), row_bcast<2>(g), row_bcast<3>(g),
                       row_bcast<4>(g), row_bcast<5>(g), row_bcast<6>(g), row_bcast<7>(g)};
#pragma unroll
  for (int j = 0; j < 8; ++j) G[j] = ACC ? __builtin_fmaf(gb[j], x[j], G[j]) : gb[j] * x[j];
}

// registers for this many waves per SIMD: what keeps the kernels from spilling (C = 3 at two
// waves: 320 bytes of scratch, 128^3 98 us against 76, 256^3 850 against 488)
__host__ __device__ constexpr int waves(int C, int BB) { return C == 1 ? (BB == 1 ? 3 : 2) : C == 2 && BB == 1 ? 2 : 1; }

// BB: right-hand sides staged together
template <typename T, int C, int BB>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(waves(C, BB), 8)))
void wgrad_kernel(const T* __restrict__ a, const T* __restrict__ cv, int B, const T* __restrict__ img, int n1, int n2,
                  int n3, float* __restrict__ partials) {
  constexpr int NQ = 27 * C + 1, NT = (NQ + 31) / 32, NO = 27 * NQ, kOneTile = 27 * C / 32;
  constexpr int kXB = BB * kXCells * 4, kIB = C * kICells * 2, kRed = 4 * 32 * 32 * 4;
  constexpr int kOnesAt = kXB + 2 * kIB, kUsed = kOnesAt + 2 * kOnes * 4;
  __shared__ __attribute__((aligned(16))) char lds[kUsed > kRed ? kUsed : kRed];
  __shared__ unsigned sh[4][2 * BB + C + 5], queue[kQueue][2];
  constexpr int kFlagA = 2 * BB + C, kFlagB = kFlagA + 1, kFlagC = kFlagA + 2, kFlagD = kFlagA + 3,
                kFlagE = kFlagA + 4;
  float* xs = (float*)lds;      // [BB][kXCells]
  f16* ih = (f16*)(lds + kXB);  // [C][kICells], then the low parts
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = lane >> 5, m = lane & 31;
  const long V = (long)n1 * n2 * n3;
  const unsigned tz = (unsigned)((n3 + kZ - 1) / kZ), tj = (unsigned)((n2 + kJ - 1) / kJ);
  const unsigned tiles = tz * tj * (unsigned)((n1 + kI - 1) / kI);
  for (int e = threadIdx.x; e < 2 * kOnes; e += kThreads)
    *(unsigned*)(lds + kOnesAt + 4 * e) = e < kOnes ? 0x3c003c00u : 0u;

  // word offsets in LDS of the lane's tap (27 .. 31 repeat tap 26, their rows are dropped)
  // and columns at row (0, w), and their steps to the row of the other half tile; the column
  // of ones stays where it is
  const int p = m < 27 ? m : 26;
  const int xo = (p / 9) * kXPlane + (p / 3 % 3) * kXRow + w * kXRow + 8 * h + p % 3;
  int io[NT], lo_o[NT], ish[NT];
  const bool one = 32 * kOneTile + m == 27 * C;
  const int on_row = one ? 0 : 1;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int q = 32 * t + m < 27 * C ? 32 * t + m : 27 * C - 1, c = q / 27, s = q % 27;
    // word of the first of the lane's cells: d3 = 0 starts on a word, d3 = -1 / +1 half a
    // word later than the word before / at it
    const int word = (c * kICells + (s / 9) * kIPlane + (s / 3 % 3) * kIRow + w * kIRow) / 2 + 4 * h + (s % 3 == 0 ? 0 : 1);
    const bool o1 = t == kOneTile && one;
    io[t] = o1 ? kOnesAt / 4 : kXB / 4 + word;
    lo_o[t] = o1 ? kOnesAt / 4 + kOnes : (kXB + kIB) / 4 + word;
    ish[t] = s % 3 == 1 ? 0 : 16;
  }
  // sums over the tiles so far
  f16x sum[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) sum[t] = f16x{};

  auto tile_at = [&](unsigned tile) {
    const unsigned u = tile / tz;
    return Pos{(int)(u / tj) * kI, (int)(u % tj) * kJ, (int)(tile % tz) * kZ};
  };
  // a row of a (range-checked: rows and cells outside the grid read 0)
  auto a_row = [&](const Pos& pos, int b, int i, int j) {
    const int gi = pos.i0 + i, gj = pos.j0 + j;
    const bool ok = gi < n1 && gj < n2 && b < B;
    return rsrc(a + (ok ? (long)b * V + ((long)gi * n2 + gj) * n3 : 0L), ok ? n3 * (int)sizeof(T) : 0);
  };
  unsigned tile = blockIdx.x;
  for (;;) {
    int queued = 0;
    for (; tile < tiles && queued < kQueue; tile += gridDim.x) {
      const Pos pos = tile_at(tile);
      // the lane's a values of a row: voxels 16 s + 8 h + lane % 8
      const unsigned go = (unsigned)(pos.z0 + 8 * h + (lane & 7)) * (unsigned)sizeof(T);
      auto load_g = [&](float (&g)[BB][4], int b0, int q) {
#pragma unroll
        for (int bb = 0; bb < BB; ++bb) {
          const auto r = a_row(pos, b0 + bb, q >> 1, w + 4 * (q & 1));
#pragma unroll
          for (int s = 0; s < 4; ++s) g[bb][s] = ld_as(r, go + 16 * s * (unsigned)sizeof(T), 0, a);
        }
      };
      bool has_lo = false;
      int ei[C];  // exponents of the image's factors
      for (int b0 = 0; b0 < B; b0 += BB) {
        Raw ri[C], rx[BB];
        if (b0 == 0) {
#pragma unroll
          for (int c = 0; c < C; ++c) load_tile(ri[c], img + c * V, pos, n1, n2, n3, w, lane);
        }
        // (an absent right-hand side repeats the last: its a reads as 0)
#pragma unroll
        for (int bb = 0; bb < BB; ++bb) load_tile(rx[bb], cv + (long)min(b0 + bb, B - 1) * V, pos, n1, n2, n3, w, lane);
        // a's rows, for the scale only (the products read them again, from L2): the two whose rows
        // of x the wave holds too, as x.m[..][u + (w == 0)]
        float rg[BB][kI * kJ / 4];
        const int rb = n3 * (int)sizeof(T), pb = n2 * rb;
        const unsigned zo = pos.z0 + lane < n3 ? (unsigned)(pos.z0 + lane) * (unsigned)sizeof(T) : kOut;
#pragma unroll
        for (int bb = 0; bb < BB; ++bb)
#pragma unroll
          for (int q = 0; q < kI * kJ / 4; ++q) {
            const int gi = pos.i0 + (q >> 1), gj = pos.j0 + ((w + 3) & 3) + 4 * (q & 1);
            const bool ok = gi < n1 && gj < n2 && b0 + bb < B;
            rg[bb][q] = ld_as(rsrc(a + (long)min(b0 + bb, B - 1) * V, ok ? n1 * pb : 0), zo, ok ? gi * pb + gj * rb : 0, a);
          }
        // largest magnitudes: c and a of each right-hand side, the image's channels
        unsigned mu[2 * BB + C], mn[C], all_v = 0, all_i = 0;
#pragma unroll
        for (int bb = 0; bb < BB; ++bb) {
          mu[2 * bb] = max_of(rx[bb]);
          float m = 0.f;
#pragma unroll
          for (int q = 0; q < kI * kJ / 4; ++q) m = max_nan(m, fabsf(rg[bb][q]));
          mu[2 * bb + 1] = magnitude(m);
          all_v = max(all_v, max(mu[2 * bb], mu[2 * bb + 1]));
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
          mu[2 * BB + c] = 0;
          if (b0 == 0) {
            all_i = max(all_i, mu[2 * BB + c] = max_of(ri[c]));
            mn[c] = min_of(ri[c]);
          }
        }
        // the largest product of a centre tap (below FP32's range it counts as none)
        float most = 0.f;
        auto centres = [&](auto first) {
#pragma unroll
          for (int bb = 0; bb < BB; ++bb)
#pragma unroll
            for (int q = 0; q < kI * kJ / 4; ++q)
              most = fmaxf(most, fabsf(rg[bb][q] * rx[bb].m[(q >> 1) + 1][(q & 1) + decltype(first)::value]));
        };
        if (w == 0) centres(std::integral_constant<int, 1>());
        else centres(std::integral_constant<int, 0>());
        const bool bad_v = __builtin_amdgcn_ballot_w64(all_v >= kInfinity) != 0;
        const bool bad_i = __builtin_amdgcn_ballot_w64(all_i >= kInfinity) != 0;
        if (bad_v || bad_i) {  // infinities set no scale
          for (int bb = 0; bb < BB; ++bb) {
            mu[2 * bb] = finite_max_of(rx[bb]);
            mu[2 * bb + 1] = 0;
            for (int q = 0; q < kI * kJ / 4; ++q) mu[2 * bb + 1] = max(mu[2 * bb + 1], finite_bits(rg[bb][q]));
          }
          for (int c = 0; c < C; ++c) mu[2 * BB + c] = b0 == 0 ? finite_max_of(ri[c]) : 0u;
        }
#pragma unroll
        for (int k = 0; k < 2 * BB + C; ++k) mu[k] = wave_max(mu[k]);
        __syncthreads();  // the previous tile's reads are done
        if (lane == 0) {
#pragma unroll
          for (int k = 0; k < 2 * BB + C; ++k) sh[w][k] = mu[k];
          sh[w][kFlagA] = (bad_v ? 1 : 0) | (bad_i ? 2 : 0);
        }
        __syncthreads();
        auto over_waves = [&](int k) {
          return (unsigned)__builtin_amdgcn_readfirstlane((int)max(max(sh[0][k], sh[1][k]), max(sh[2][k], sh[3][k])));
        };
        auto any_wave = [&](int k) {
          return (unsigned)__builtin_amdgcn_readfirstlane((int)(sh[0][k] | sh[1][k] | sh[2][k] | sh[3][k]));
        };
        const unsigned bad = any_wave(kFlagA);
        if (b0 == 0) {
#pragma unroll
          for (int c = 0; c < C; ++c) ei[c] = scale_exp(over_waves(2 * BB + c), kTargetP);
        }
        // G in units of 2^-e, the largest that a right-hand side's own factors give (they add up
        // in G; one of zeros has no say, and one 2^100 below the other adds nothing)
        int ex[BB], e = 2 * 126;
        bool some[BB];
#pragma unroll
        for (int bb = 0; bb < BB; ++bb) {
          const unsigned bx = over_waves(2 * bb), bg = over_waves(2 * bb + 1);
          ex[bb] = scale_exp(bx, kTargetG);
          some[bb] = bx != 0u && bg != 0u;
          if (some[bb]) e = min(e, ex[bb] + scale_exp(bg, kTargetG));
        }
        float sg[BB];
#pragma unroll
        for (int bb = 0; bb < BB; ++bb) sg[bb] = some[bb] && e - ex[bb] >= -126 ? pow2(e - ex[bb]) : 0.f;
#pragma unroll
        for (int bb = 0; bb < BB; ++bb) {
          const float sx = pow2(ex[bb]);
          each(rx[bb], w, lane, [&](int k, int j, int z, float v) {
            xs[bb * kXCells + k * kXPlane + j * kXRow + z] = v * sx;
          });
        }
        unsigned flags = 0;  // 1: low parts, 2: small image values, 4: a product near the bound
        flags |= __builtin_amdgcn_ballot_w64(most >= ldexpf(0.25f, -e)) != 0 ? 4u : 0u;
        if (b0 == 0) {
          unsigned any = 0;
          bool small = false;
#pragma unroll
          for (int c = 0; c < C; ++c) {
            const float si = pow2(ei[c]);
            small |= mn[c] < least_bits(ei[c]);
            each(ri[c], w, lane, [&](int k, int j, int z, float v) {
              const float sv = v * si;
              const f16 hi = (f16)sv, lo = (f16)(sv - (float)hi);
              f16* d = ih + c * kICells + k * kIPlane + j * kIRow + 1 + z;
              d[0] = hi;
              d[C * kICells] = lo;
              any |= __builtin_bit_cast(unsigned short, lo);
            });
          }
          flags |= __builtin_amdgcn_ballot_w64((any & 0x7fffu) != 0) != 0 ? 1u : 0u;
          flags |= __builtin_amdgcn_ballot_w64(small) != 0 ? 2u : 0u;
        }
        if (lane == 0) sh[w][kFlagB] = flags;
        __syncthreads();
        flags = any_wave(kFlagB);
        if (b0 == 0) has_lo = (flags & 1) != 0;
        // (an image that does not do sends all of the tile's right-hand sides to the queue)
        bool wide = bad != 0;
        if (b0 == 0 && !wide && (flags & 2)) {
          bool rows = false;
#pragma unroll 1
          for (int c = 0; c < C; ++c) {
            Raw r;  // (read again: kept, the cells would take registers from everyone)
            load_tile(r, img + c * V, pos, n1, n2, n3, w, lane);
            int ec = ei[0];
#pragma unroll
            for (int k = 1; k < C; ++k) ec = c == k ? ei[k] : ec;
            rows |= has_small_rows(r, img + c * V, pos, n1, n2, n3, least_bits(ec));
          }
          const bool any = __builtin_amdgcn_ballot_w64(rows) != 0;
          if (lane == 0) sh[w][kFlagC] = any;
          __syncthreads();
          wide = any_wave(kFlagC) != 0;
        }
        const bool none = e == 2 * 126;  // no right-hand side has both x and g
        if (none && !wide) continue;
        if (!wide && !(flags & 4)) {
          // no centre tap comes near the bound (x may be large beside a solid, where g lies in it):
          // G's own largest value sets its scale
          float top = 0.f;
          unsigned pairs = 0;
#pragma unroll 1
          for (int q = 0; q < kI * kJ / 4; ++q) {
            const int pi = q >> 1, pj = w + 4 * (q & 1);
#pragma unroll
            for (int bb = 0; bb < BB; ++bb) {
              const float g = ld_as(a_row(pos, b0 + bb, pi, pj), (unsigned)(pos.z0 + lane) * (unsigned)sizeof(T), 0, a);
#pragma unroll 1
              for (int d = 0; d < 9; ++d) {
                const float* x = xs + bb * kXCells + (pi + d / 3) * kXPlane + (pj + d % 3) * kXRow + lane;
                const float m = fmaxf(fabsf(x[0]), fmaxf(fabsf(x[1]), fabsf(x[2])));
                top = fmaxf(top, fabsf(g * sg[bb]) * m);
                pairs |= g != 0.f && m != 0.f;
              }
            }
          }
          const unsigned m = wave_max(__float_as_uint(top));
          const bool some_g = __builtin_amdgcn_ballot_w64(pairs != 0) != 0;
          if (lane == 0) {
            sh[w][kFlagD] = m;
            sh[w][kFlagE] = some_g;
          }
          __syncthreads();
          const unsigned most_g = over_waves(kFlagD);
          if (any_wave(kFlagE) == 0) continue;
          const int up = 2 * kTargetG + 1 - exponent_of(most_g);
          wide = most_g == 0u;
#pragma unroll
          for (int bb = 0; bb < BB; ++bb) {
            if (!some[bb]) continue;
            wide |= e + up - ex[bb] > 126;
            sg[bb] = e + up - ex[bb] >= -126 ? pow2(min(e + up - ex[bb], 126)) : 0.f;
          }
          e += up;
        }
        if (wide) {
          if (threadIdx.x == 0) {
            queue[queued][0] = tile;
            queue[queued][1] = (unsigned)b0;
          }
          ++queued;
          break;
        }
        // the products of the high parts, and those with a low part
        f16x acc[NT], acl[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = acl[t] = f16x{};

        auto rows = [&](auto lo_c) {
          constexpr bool LO = decltype(lo_c)::value;
          // operands of one product step, read one step ahead of their use
          struct Step {
            float x[BB][8];
            unsigned ph[NT][5];
          };
          struct Base {
            int x, i[NT], l[NT];
          };
          auto base = [&](int q) {  // row w + 4 (q % 2) of plane q / 2
            const int irow = ((q >> 1) * kIPlane + (q & 1) * 4 * kIRow) / 2;
            Base r;
            r.x = xo + (q >> 1) * kXPlane + (q & 1) * 4 * kXRow;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
              const int step = t == kOneTile ? on_row * irow : irow;
              r.i[t] = io[t] + step;
              r.l[t] = lo_o[t] + step;
            }
            return r;
          };
          auto load = [&](Step& st, const Base& r, int s) {
#pragma unroll
            for (int bb = 0; bb < BB; ++bb)
#pragma unroll
              for (int j = 0; j < 8; ++j) st.x[bb][j] = ((const float*)lds)[r.x + bb * kXCells + 16 * s + j];
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
              for (int k = 0; k < 5; ++k) st.ph[t][k] = ((const unsigned*)lds)[r.i[t] + 8 * s + k];
          };
          float gc[BB][4], gn[BB][4];
          load_g(gc, b0, 0);
          Base bc = base(0);
          Step cur;
          load(cur, bc, 0);
#pragma unroll 1
          for (int q = 0; q < kI * kJ / 4; ++q) {
            const int qn = q + 1 < kI * kJ / 4 ? q + 1 : q;
            load_g(gn, b0, qn);
            const Base bn = base(qn);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
              Step nxt;
              if (s < 3) load(nxt, bc, s + 1);
              else load(nxt, bn, 0);
              float G[8];
#pragma unroll
              for (int bb = 0; bb < BB; ++bb) {
                if (bb == 0) products<false>(gc[bb][s] * sg[bb], cur.x[bb], G);
                else products<true>(gc[bb][s] * sg[bb], cur.x[bb], G);
              }
              u32x4s gh, gl;
#pragma unroll
              for (int k = 0; k < 4; ++k) {
                unsigned hi, lo;
                split_pair(G[2 * k], G[2 * k + 1], hi, lo);
                gh[k] = hi;
                gl[k] = lo;
              }
              auto cols = [&](const unsigned (&x)[5], int t) {
                u32x4s r;
#pragma unroll
                for (int k = 0; k < 4; ++k) r[k] = __builtin_amdgcn_alignbit(x[k + 1], x[k], (unsigned)ish[t]);
                return __builtin_bit_cast(h8, r);
              };
              const h8 ah = __builtin_bit_cast(h8, gh), al = __builtin_bit_cast(h8, gl);
#pragma unroll
              for (int t = 0; t < NT; ++t) {
                const h8 ph = cols(cur.ph[t], t);
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, ph, acc[t], 0, 0, 0);
                acl[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, ph, acl[t], 0, 0, 0);
                if (LO) {
                  unsigned pl[5];
#pragma unroll
                  for (int k = 0; k < 5; ++k) pl[k] = ((const unsigned*)lds)[bc.l[t] + 8 * s + k];
                  acl[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, cols(pl, t), acl[t], 0, 0, 0);
                }
              }
              cur = nxt;
            }
            bc = bn;
#pragma unroll
            for (int bb = 0; bb < BB; ++bb)
#pragma unroll
              for (int s = 0; s < 4; ++s) gc[bb][s] = gn[bb][s];
          }
        };
        if (has_lo) rows(std::true_type());
        else rows(std::false_type());
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          int u = -e;  // the column's scale: of G, and of the image's channel
#pragma unroll
          for (int c = 0; c < C; ++c) u -= (32 * t + m) / 27 == c && 32 * t + m < 27 * C ? ei[c] : 0;
#pragma unroll
          for (int i = 0; i < 16; ++i) sum[t][i] += ldexpf(acc[t][i] + acl[t][i], u);
        }
      }
    }
    if (queued == 0) break;
    // FP32 products of the tiles that wait, from their first right-hand side that has to
    int hv = h, mv = m;  // opaque: nothing of this is to be worked out before, or kept in registers
    asm volatile("" : "+v"(hv), "+v"(mv));
    int col[NT], off[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int p0 = 8 * (i >> 2) + (i & 3), p1 = p0 + 4 < 27 ? p0 + 4 : 26, tap = hv ? p1 : p0;
      off[i] = (tap / 9) * kXPlane + (tap / 3 % 3) * kXRow + tap % 3;
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int q = min(32 * t + mv, 27 * C - 1), s = q % 27;
      col[t] = (q / 27) * kICells + (s / 9) * kIPlane + (s / 3 % 3) * kIRow + 1 + s % 3;
    }
#pragma unroll 1
    for (int k = 0; k < queued; ++k) {
      __syncthreads();
      const Pos pos = tile_at((unsigned)__builtin_amdgcn_readfirstlane((int)queue[k][0]));
#pragma unroll 1
      for (int c = 0; c < C; ++c) {  // the image as it is, in the space of its two parts
        Raw r;
        load_tile(r, img + c * V, pos, n1, n2, n3, w, lane);
        each(r, w, lane, [&](int k, int j, int z, float v) {
          ((float*)ih)[c * kICells + k * kIPlane + j * kIRow + 1 + z] = v;
        });
      }
#pragma unroll 1
      for (int b = __builtin_amdgcn_readfirstlane((int)queue[k][1]); b < B; ++b) {
        Raw r;
        load_tile(r, cv + (long)b * V, pos, n1, n2, n3, w, lane);
        __syncthreads();
        each(r, w, lane, [&](int k, int j, int z, float v) { xs[k * kXPlane + j * kXRow + z] = v; });
        __syncthreads();
#pragma unroll 1
        for (int q = 0; q < kI * kJ / 4; ++q) {
          const int pi = q >> 1, pj = w + 4 * (q & 1), gi = pos.i0 + pi, gj = pos.j0 + pj;
          if (gi >= n1 || gj >= n2) continue;
          const float ga = ld_as(a_row(pos, b, pi, pj), (unsigned)(pos.z0 + lane) * (unsigned)sizeof(T), 0, a);
          f16x row[NT];
#pragma unroll
          for (int t = 0; t < NT; ++t) row[t] = f16x{};
#pragma unroll 1
          for (int z = 0; z < min(kZ, n3 - pos.z0); ++z) {
            const float av = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ga), z));
            const int at = pi * kXPlane + pj * kXRow + z;
            float pv[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
              const float v = ((const float*)ih)[col[t] + pi * kIPlane + pj * kIRow + z];
              pv[t] = 32 * t + mv >= 27 * C ? 1.f : v;
            }
            if (magnitude(av) < kInfinity) {  // (beyond the grid x is 0)
#pragma unroll
              for (int i = 0; i < 16; ++i) {
                const float G = av * xs[off[i] + at];
#pragma unroll
                for (int t = 0; t < NT; ++t) row[t][i] = fmaf(G, pv[t], row[t][i]);
              }
              continue;
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              asm volatile("" : "+v"(hv));
              const int p0 = 8 * (i >> 2) + (i & 3), p1 = p0 + 4 < 27 ? p0 + 4 : 26, tap = hv ? p1 : p0;
              const bool in = (unsigned)(gi + tap / 9 - 1) < (unsigned)n1 && (unsigned)(gj + tap / 3 % 3 - 1) < (unsigned)n2 &&
                              (unsigned)(pos.z0 + z + tap % 3 - 1) < (unsigned)n3;
              const float G = av * xs[off[i] + at];
#pragma unroll
              for (int t = 0; t < NT; ++t) row[t][i] = fmaf(in ? G : 0.f, pv[t], row[t][i]);
            }
          }
#pragma unroll
          for (int t = 0; t < NT; ++t) sum[t] += row[t];
        }
      }
    }
  }
  // D[8 (i / 4) + 4 h + i % 4][32 t + m] of the wave, the waves added in order
  float* red = (float*)lds;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i)
      red[(w * 32 + 8 * (i >> 2) + 4 * h + (i & 3)) * 32 + m] = sum[t][i];
    __syncthreads();
    for (int e = threadIdx.x; e < 27 * 32; e += kThreads) {
      const int pp = e >> 5, q = 32 * t + (e & 31);
      if (q < NQ)
        partials[(size_t)blockIdx.x * NO + pp * NQ + q] =
            (red[e] + red[1024 + e]) + (red[2048 + e] + red[3072 + e]);
    }
  }
}

// workgroups: one per tile, at most `most` (the partial sums' workspace)
inline int blocks(int most, int n1, int n2, int n3) {
  const long tiles = (long)((n1 + kI - 1) / kI) * ((n2 + kJ - 1) / kJ) * ((n3 + kZ - 1) / kZ);
  return (int)(tiles < most ? tiles : most);
}

template <typename T>
void launch(const void* a, const void* c, const void* img, float* part, int nblk, int C, int B, int n1, int n2, int n3,
            hipStream_t st) {
#define MLPCG_WGK(CC)                                                                                               \
  if (C == CC) {                                                                                                    \
    if (B == 1)                                                                                                     \
      wgrad_kernel<T, CC, 1><<<nblk, kThreads, 0, st>>>((const T*)a, (const T*)c, B, (const T*)img, n1, n2, n3, part); \
    else                                                                                                            \
      wgrad_kernel<T, CC, 2><<<nblk, kThreads, 0, st>>>((const T*)a, (const T*)c, B, (const T*)img, n1, n2, n3, part); \
  }
  MLPCG_WGK(1) MLPCG_WGK(2) MLPCG_WGK(3)
#undef MLPCG_WGK
}

}  // namespace wgrad

int wgrad_blocks(int most, int n1, int n2, int n3) { return wgrad::blocks(most, n1, n2, n3); }

int launch_wgrad(int dtype, const void* a, const void* c, const void* img, float* part, int nblk, int C, int B, int n1,
                 int n2, int n3, hipStream_t st) {
  MLPCG_REQUIRE((long)n1 * n2 * n3 * (dtype == kF32 ? 4 : 2) < (1L << 31), "weight_grad: grid (%d,%d,%d) too large", n1,
                n2, n3);
  if (dtype == kF32) wgrad::launch<float>(a, c, img, part, nblk, C, B, n1, n2, n3, st);
  else if (dtype == kF16) wgrad::launch<f16>(a, c, img, part, nblk, C, B, n1, n2, n3, st);
  else if (dtype == kBF16) wgrad::launch<bf16>(a, c, img, part, nblk, C, B, n1, n2, n3, st);
  else MLPCG_REQUIRE(false, "weight_grad: bad dtype %d", dtype);
  return check_launch("weight_grad");
}

}  // namespace mlpcg
