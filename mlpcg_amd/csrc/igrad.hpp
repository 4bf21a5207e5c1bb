// Input gradient of an SM block, the adjoint of split.hpp's apply:
//
//   dx(u) = sum_p K_p(u - d_p) g(u - d_p)
//
// (sm_block_3d_kernel.cu:231-260), K as in split.hpp: recomputed on the matrix cores, neither
// stored nor streamed.  A lane holds K of both z parities for the taps of its columns, so the
// products K_p(v) g(v) are formed where K is made and summed along the way:
//   * along z in the lane (the two parities of a pair) and once per row over DPP, for the cells
//     that the neighbouring lanes' pairs reach;
//   * along j by marching: a wave takes one plane and walks its source rows j0 - 1 .. j0 + R,
//     with the sums of the rows j - 1, j, j + 1 of its columns in registers;
//   * along i through memory: T[d1](i, j, k), d1 = -1, 0, +1, is what plane i adds to plane
//     i + d1; the gather kernel adds the three.  The cells that a tile's first and last lane
//     add to the neighbouring z tiles go to a side array, an entry per row and tile.
// The lower lanes hold the columns of d1 = -1 and two of d1 = 0, the upper lanes those of
// d1 = +1 and the third of d1 = 0 (its row j + 1, while the lower lanes finish row j - 1 from
// theirs: the upper lanes' sums wait two steps).  All sums are FP32 in a fixed order.  Tiles
// and blocks that ask for exact stencils get them as in split.hpp.
#pragma once

#include <algorithm>

#include "kernels.hpp"
#include "split.hpp"

namespace mlpcg {
namespace split {

constexpr int kIgPlanes = 4;  // planes per tile, one per wave
// Output rows per tile, R: the march computes R + 2 rows of K for R of dx, so long marches cost
// less (256^3), but a small grid needs more workgroups than they leave (64^3: 64 of 16 rows).
__host__ __device__ constexpr int ig_rows(int C) { return C == 1 ? 16 : 8; }
// registers for this many waves per SIMD (C = 3 without its 52 to 84 bytes of scratch leaves one
// wave: 128^3 82 us against 63)
__host__ __device__ constexpr int ig_waves(int C, int BB) { return C == 1 && BB == 1 ? 3 : 2; }

constexpr unsigned kIgBlocks = 512;

struct IgradArgs {
  const void* img;   // [C][V]
  const void* pack;  // launch_split_pack
  const void* g;     // [B][V]
  float* T;          // [B][3][V], d1 = -1, 0, +1
  float* edge;       // [B][n1][n2][z tiles][4][2]
  int B, n1, n2, n3;
};

// sums of one row: even and odd cell of the lane's pair, and what it adds to the even cell of
// the next lane and the odd cell of the previous one
struct RowSum {
  float e, o, ex, ox;
};
__device__ __forceinline__ void add_column(RowSum& s, const float (&ke)[3], const float (&ko)[3], float ge, float go) {
  s.e = fmaf(ko[0], go, fmaf(ke[1], ge, s.e));
  s.o = fmaf(ke[2], ge, fmaf(ko[1], go, s.o));
  s.ex = fmaf(ko[2], go, s.ex);
  s.ox = fmaf(ke[0], ge, s.ox);
}

__device__ __forceinline__ void store_pair(float* p, float a, float b, bool ok0, bool ok1, bool pair) {
  if (pair && ok1) {
    *(float2*)p = float2{a, b};
  } else {
    if (ok0) p[0] = a;
    if (ok1) p[1] = b;
  }
}

template <typename TI, int C, int R, int BB>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(ig_waves(C, BB), 8)))
void igrad_kernel(IgradArgs a) {
  constexpr int PJ = R + 4, FI = kIgPlanes, kCells = tile_cells(FI, PJ);
  constexpr bool FULL = sizeof(TI) == 4;
  __shared__ __attribute__((aligned(16))) char im[C * kCells * (FULL ? 4 : 2)];
  __shared__ unsigned sh[4 * (C + 2)];
  const f16 *ih = (const f16*)im, *il = ih + C * kCells;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = lane >> 5, n = lane & 31;
  const unsigned tz = (unsigned)((a.n3 + kZ - 1) / kZ), tj = (unsigned)((a.n2 + R - 1) / R);
  const unsigned t = xcd_block(blockIdx.x, gridDim.x), u = t / tz;
  const int i0 = (int)(u / tj) * FI, j0 = (int)(u % tj) * R, zt = (int)(t % tz), z0 = zt * kZ;
  const long plane = (long)a.n2 * a.n3, V = a.n1 * plane;
  const int b0 = blockIdx.y * BB;

  Raw<FI, PJ> ri[C];
#pragma unroll
  for (int c = 0; c < C; ++c)
    load_raw<FI, PJ>(ri[c], (const TI*)a.img + c * V, Tile{i0, j0 - 1, z0}, a.n1, a.n2, a.n3, w, lane);
  const PackHeader* hd = (const PackHeader*)a.pack;
  const ImageTile<C> it =
      stage_image<TI, C, FI, PJ>(ri, hd, 0, 0, w, lane, im, sh, (const TI*)a.img, Tile{i0, j0 - 1, z0}, a.n1, a.n2, a.n3);
  const int i = i0 + w;
  if (i >= a.n1) return;  // uniform; no barrier follows
  Weights<C> W;
  W.load(a.pack, lane);
  W.set_bias(ldexpf(((const float*)((const char*)a.pack + kHeaderBytes + pack_w_bytes(C)))[lane & 31], it.E - kOne), h);
  WordBase wb;
  wb.init<PJ>(h, n, w * PJ);

  const bool ok0 = z0 + 2 * n < a.n3, ok1 = z0 + 2 * n + 1 < a.n3, ragged = z0 + kZ > a.n3, pair = (a.n3 & 1) == 0;
  constexpr unsigned kSize = (unsigned)sizeof(TI);
  const unsigned o0 = ok0 ? (unsigned)(z0 + 2 * n) * kSize : 0x80000000u;
  const unsigned o1 = ok1 ? (unsigned)(z0 + 2 * n + 1) * kSize : 0x80000000u;
  const int pb = (int)(plane * (int)kSize), rb = a.n3 * (int)kSize;
  float gn[BB][2];  // the next row's g
  auto load_g = [&](int j) {
    const bool in = (unsigned)j < (unsigned)a.n2;
#pragma unroll
    for (int bb = 0; bb < BB; ++bb) {
      const bool ok = in && (BB == 1 || b0 + bb < a.B);
      const TI* gp = (const TI*)a.g + (ok ? (long)(b0 + bb) * V + i * plane : 0);
      const auto r = rsrc(gp, ok ? pb : 0);
      gn[bb][0] = ld_as(r, o0, ok ? j * rb : 0, gp);
      gn[bb][1] = ld_as(r, o1, ok ? j * rb : 0, gp);
    }
  };
  const int rows = min(R, a.n2 - j0);  // output rows
  const long e8 = (long)tz * 8;

  // Returns whether a sum is infinite or NaN.  (K scaled by 2^E overflows where g is some 2^90 or
  // more: the wave then marches again with exact stencils.)
  auto march = [&](auto mode) -> bool {
    constexpr int M = decltype(mode)::value;  // 0: hi alone, 1: hi and lo, 2: exact stencils
    const int back = M == 2 ? 0 : -it.E;
    float most = 0.f;
    RowSum m[BB][3], q[BB][2];
    float d1[BB][2], d2[BB][2];
#pragma unroll
    for (int bb = 0; bb < BB; ++bb) {
#pragma unroll
      for (int k = 0; k < 3; ++k) m[bb][k] = RowSum{0.f, 0.f, 0.f, 0.f};
      q[bb][0] = q[bb][1] = RowSum{0.f, 0.f, 0.f, 0.f};
      d1[bb][0] = d1[bb][1] = d2[bb][0] = d2[bb][1] = 0.f;
    }
    load_g(j0 - 1);
    // where the lane's pair, its cell of T[0] and its edge sums of row j - 1 go; one row on per step
    float *pm[BB], *pq[BB];
    float* pe[BB];
#pragma unroll
    for (int bb = 0; bb < BB; ++bb) {
      float* T = a.T + (long)(b0 + bb) * 3 * V + i * plane + (long)(j0 - 2) * a.n3 + z0 + 2 * n;
      pm[bb] = T + (h ? 2 * V : 0);
      pq[bb] = T + V + h;
      // [row][z tile][main, mid of the lower / upper lanes][right, left]
      pe[bb] = a.edge + (((long)(b0 + bb) * a.n1 + i) * a.n2 + j0 - 2) * e8 + zt * 8 + 2 * h + (n == 0 ? 1 : 0);
    }
#pragma unroll 1
    for (int s = 0; s < rows + 2; ++s) {
      const int j = j0 - 1 + s;
      float g[BB][2];
#pragma unroll
      for (int bb = 0; bb < BB; ++bb) {
        g[bb][0] = gn[bb][0];
        g[bb][1] = gn[bb][1];
      }
      load_g(j + 1);
      if ((unsigned)j < (unsigned)a.n2) {  // uniform
        f16x K[2];
        if constexpr (M == 2)
          exact_stencils<C, PJ>(a.pack, kCells, (w * PJ + s) * kPitch + 2 * n, h, K, [&](int c, int e) {
            if (it.exact) return (float)((const TI*)im)[e];  // uniform
            int fc = it.f[0];
#pragma unroll
            for (int k = 1; k < C; ++k) fc = c == k ? it.f[k] : fc;
            return ldexpf((float)ih[e] + (FULL ? (float)il[e] : 0.f), -fc);
          });
        else
          stencils<C, M == 1, C != 3 || M == 1>(W, ih, il, kCells, wb, s * kPitch, K);
        if (ragged) {  // uniform: cells past the grid add nothing, whatever K is there
#pragma unroll
          for (int k = 0; k < 15; ++k) {
            K[0][k] = ok0 ? K[0][k] : 0.f;
            K[1][k] = ok1 ? K[1][k] : 0.f;
          }
        }
#pragma unroll
        for (int bb = 0; bb < BB; ++bb) {
#pragma unroll
          for (int c = 0; c < 5; ++c) {
            const float ke[3] = {K[0][3 * c], K[0][3 * c + 1], K[0][3 * c + 2]};
            const float ko[3] = {K[1][3 * c], K[1][3 * c + 1], K[1][3 * c + 2]};
            add_column(c < 3 ? m[bb][c < 3 ? c : 0] : q[bb][c == 3 ? 0 : 1], ke, ko, g[bb][0], g[bb][1]);
          }
        }
      }
      // rows j - 1 (and j + 1 of the upper lanes' column of d1 = 0) are complete
      const bool out = s >= 2, mid1 = s < rows;
#pragma unroll
      for (int bb = 0; bb < BB; ++bb) {
        if (BB > 1 && b0 + bb >= a.B) break;
        RowSum r = m[bb][0], p = q[bb][0];
        r = RowSum{ldexpf(r.e, back), ldexpf(r.o, back), ldexpf(r.ex, back), ldexpf(r.ox, back)};
        p = RowSum{ldexpf(p.e, back), ldexpf(p.o, back), ldexpf(p.ex, back), ldexpf(p.ox, back)};
        if (M != 2) {
          most = max_nan(most, max_nan(fabsf(r.e), fabsf(r.o)));
          most = max_nan(most, max_nan(fabsf(r.ex), fabsf(r.ox)));
          most = max_nan(most, max_nan(fabsf(p.e), fabsf(p.o)));
          most = max_nan(most, max_nan(fabsf(p.ex), fabsf(p.ox)));
        }
        // (all lanes take part in the shifts; the first or last of a half drops what it received)
        const float rx = wave_from_prev(r.ex), ry = wave_from_next(r.ox);
        const float px = wave_from_prev(p.ex), py = wave_from_next(p.ox);
        const float re = r.e + (n == 0 ? 0.f : rx), ro = r.o + (n == 31 ? 0.f : ry);
        const float qe = p.e + (n == 0 ? 0.f : px), qo = p.o + (n == 31 ? 0.f : py);
        const float mid = halves_sum(h ? d2[bb][0] : qe, h ? d2[bb][1] : qo);
        if (out) {
          store_pair(pm[bb], re, ro, ok0, ok1, pair);
          if (h ? ok1 : ok0) *pq[bb] = mid;
        }
        if (n == 31 || n == 0) {
          if (out) pe[bb][0] = n == 0 ? r.ox : r.ex;
          if (h ? mid1 : out) pe[bb][4 + (h ? 2 * e8 : 0)] = n == 0 ? p.ox : p.ex;
        }
        pm[bb] += a.n3;
        pq[bb] += a.n3;
        pe[bb] += e8;
        m[bb][0] = m[bb][1];
        m[bb][1] = m[bb][2];
        m[bb][2] = RowSum{0.f, 0.f, 0.f, 0.f};
        // (the upper lanes' fifth column is a dummy: 0 times an infinity must not stay)
        q[bb][0] = h ? RowSum{0.f, 0.f, 0.f, 0.f} : q[bb][1];
        q[bb][1] = RowSum{0.f, 0.f, 0.f, 0.f};
        d2[bb][0] = d1[bb][0];
        d2[bb][1] = d1[bb][1];
        d1[bb][0] = qe;
        d1[bb][1] = qo;
      }
    }
    return __builtin_amdgcn_ballot_w64(magnitude(most) >= kInfinity) != 0;
  };
  bool exact = it.exact;
  if (!exact) exact = FULL && it.has_lo ? march(std::integral_constant<int, FULL ? 1 : 0>()) : march(std::integral_constant<int, 0>());
  if (exact) march(std::integral_constant<int, 2>());
}

// dx(i, j, k) = T[-1](i + 1) + T[0](i) + T[+1](i - 1), plus the z tiles' edge sums
template <typename TY, int VZ>
__global__ __launch_bounds__(kThreads) void igrad_gather_kernel(const float* __restrict__ T, const float* __restrict__ edge,
                                                                TY* __restrict__ dx, int n1, int n2, int n3) {
  const long plane = (long)n2 * n3, V = n1 * plane;
  const long c = (long)xcd_block(blockIdx.x, gridDim.x) * kThreads + threadIdx.x, v = c * VZ;
  if (v >= V) return;
  T += (long)blockIdx.y * 3 * V;
  dx += (long)blockIdx.y * V;
  const long row = v / n3;
  const int k = (int)(v - row * n3), i = (int)(row / n2);
  float s[VZ], q[VZ];
  load_vec_nt<VZ>(T + V + v, s);
  if (i + 1 < n1) {
    load_vec_nt<VZ>(T + v + plane, q);
#pragma unroll
    for (int t = 0; t < VZ; ++t) s[t] += q[t];
  }
  if (i > 0) {
    load_vec_nt<VZ>(T + 2 * V + v - plane, q);
#pragma unroll
    for (int t = 0; t < VZ; ++t) s[t] += q[t];
  }
  const int tz = (n3 + kZ - 1) / kZ;
  auto add = [&](int zt, int side) {
    const float* e = edge + (((long)blockIdx.y * n1 * n2 + row) * tz + zt) * 8 + side;
    float r = e[4] + e[6];
    if (i + 1 < n1) r += e[(long)n2 * tz * 8];
    if (i > 0) r += e[-(long)n2 * tz * 8 + 2];
    return r;
  };
  if (k % kZ == 0 && k > 0) s[0] += add(k / kZ - 1, 0);
  if ((k + VZ) % kZ == 0 && k + VZ < n3) s[VZ - 1] += add((k + VZ) / kZ, 1);
  store_vec<VZ>(dx + v, s);
}

template <typename TI, int C>
void launch_igrad_c(const IgradArgs& a, hipStream_t st) {
  auto blocks = [&](int R) {
    return (unsigned)((a.n1 + kIgPlanes - 1) / kIgPlanes) * (unsigned)((a.n2 + R - 1) / R) * (unsigned)((a.n3 + kZ - 1) / kZ);
  };
  auto run = [&](auto r) {
    constexpr int R = decltype(r)::value;
    if (a.B == 1) igrad_kernel<TI, C, R, 1><<<dim3(blocks(R), 1), kThreads, 0, st>>>(a);
    else igrad_kernel<TI, C, R, 2><<<dim3(blocks(R), (unsigned)((a.B + 1) / 2)), kThreads, 0, st>>>(a);
  };
  if (blocks(ig_rows(C)) >= kIgBlocks) run(std::integral_constant<int, ig_rows(C)>());
  else run(std::integral_constant<int, 4>());
}

template <typename TI>
int launch_igrad_t(const void* img, const void* pack, const TI* g, TI* dx, void* work, size_t bytes, int C, int B, int n1,
                   int n2, int n3, hipStream_t st) {
  const size_t V = (size_t)n1 * n2 * n3;
  const int most = (int)std::min<size_t>(bytes / fused_sgrad_bytes(n1, n2, n3), 65535);
  MLPCG_REQUIRE(most >= 1, "igrad: workspace of %zu bytes is too small", bytes);
  for (int b = 0; b < B; b += most) {
    const int nb = std::min(most, B - b);
    IgradArgs a;
    a.img = img;
    a.pack = pack;
    a.g = g + (size_t)b * V;
    a.T = (float*)work;
    a.edge = (float*)((char*)work + (((size_t)nb * 3 * V * sizeof(float) + 255) & ~(size_t)255));
    a.B = nb;
    a.n1 = n1;
    a.n2 = n2;
    a.n3 = n3;
    if (C == 1) launch_igrad_c<TI, 1>(a, st);
    else if (C == 2) launch_igrad_c<TI, 2>(a, st);
    else launch_igrad_c<TI, 3>(a, st);
    const int vz = n3 % 4 == 0 ? 4 : 1;
    const dim3 gr((unsigned)((V / vz + kThreads - 1) / kThreads), (unsigned)nb);
    if (vz == 4) igrad_gather_kernel<TI, 4><<<gr, kThreads, 0, st>>>((const float*)work, a.edge, dx + (size_t)b * V, n1, n2, n3);
    else igrad_gather_kernel<TI, 1><<<gr, kThreads, 0, st>>>((const float*)work, a.edge, dx + (size_t)b * V, n1, n2, n3);
  }
  return check_launch("igrad");
}

}  // namespace split

size_t fused_sgrad_bytes(int n1, int n2, int n3) {
  const size_t rows = (size_t)n1 * n2;
  return ((3 * rows * n3 * sizeof(float) + 255) & ~(size_t)255) +
         rows * ((n3 + split::kZ - 1) / split::kZ) * 8 * sizeof(float) + 256;
}

// Time of launch_igrad and the packing, stored K and its transposed gather -> now: FP32 C = 1
// 256^3 835 -> 216 us, 128^3 98 -> 39 us, two right-hand sides 119 -> 55 us, 64^3 25 -> 18 us;
// C = 3 256^3 1730 -> 468 us; BF16 256^3 C = 1 280 (nine BF16 column sums) -> 180 us, C = 3 409 ->
// 360 us.  Errors against 64 bits (norm-wise): FP32 0.9 to 1.3e-7 (was 1.0 to 1.9e-7), BF16
// 1.7e-3, the result's rounding (was 2.1 to 2.5e-3).
int launch_igrad(int dtype, const void* img, const void* pack, const void* g, void* dx, void* work, size_t bytes, int C,
                 int B, int n1, int n2, int n3, hipStream_t st) {
  MLPCG_REQUIRE(split_eligible(C, n1, n2, n3), "igrad: grid (%d,%d,%d) / C=%d not supported", n1, n2, n3, C);
  MLPCG_REQUIRE(dtype == kF32 || dtype == kBF16, "igrad: bad dtype %d", dtype);
  if (dtype == kBF16)
    return split::launch_igrad_t<bf16>(img, pack, (const bf16*)g, (bf16*)dx, work, bytes, C, B, n1, n2, n3, st);
  return split::launch_igrad_t<float>(img, pack, (const float*)g, (float*)dx, work, bytes, C, B, n1, n2, n3, st);
}

}  // namespace mlpcg
