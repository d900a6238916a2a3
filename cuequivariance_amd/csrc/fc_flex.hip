// Fully connected product with shared weights and a second operand of multiplicity one (uvw,iu,jv,kw+ijk, v = 1), table-driven:
//
//   out[z, k, w] = sum over the paths p of the block   sum_ij C_p[i, j, k] x2[z, j] sum_u x1[z, i, u] W_p[u, w]
//
// In the manner of linear_flex.hip: a wavefront takes 32 rows x 32 columns of one result block (all its components), weights and
// rows straight from the caches, no LDS for operands, no barriers.  The products are issued as W-columns x rows, so a lane holds one
// row: T_i = x1_i W_p stays in registers, and the factors s_ik = sum_j C_p[i, j, k] x2[z, j] are scalars of the lane:
// acc_k += s_ik T_i.  The input gradient is the same kernel on the cotangent with W_p read transposed and the coefficients
// transposed; the gradient of x2 needs the same products R_k = W_p g_k against x1 and is formed there too: per-lane dot products,
// summed over the paths in a small LDS array, one partial row per column tile, folded in order.  The weight gradient contracts the
// rows: x1_i against H_i = sum_k s_ik g_k formed in registers.
//
// Why not the generated kernels (codegen/fullyconnected.py: a wavefront per 32 rows and ALL columns, weights in LDS) for every size:
// their unit is 19 us long for 64x0e+64x1o, a few thousand rows leave most of the chip idle and 50 000 rows are 0.76 of a round.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "cw_common.h"
#include "u1d_spec.h"

namespace cueq {
namespace {

struct FcPart {          // one path: its weights, the source block it contracts, its factors
  int64_t w0;
  int32_t a0, K, D, coef;  // source block: offset, multiplicity, components; coef: offset of the D x DR x d2 factors
  int32_t j0, d2;
  int32_t stride, unused;  // elements between weight rows as stored
};
struct FcBlock {  // one block of the result
  int32_t c0, N, D, first, parts, nt;
};

typedef float fx16 __attribute__((ext_vector_type(16)));

template <typename TI>
__device__ __forceinline__ float fc_widen(const TI* p) {
  if constexpr (sizeof(TI) == 4) return *reinterpret_cast<const float*>(p);
  else return mm_widen<TI>(*reinterpret_cast<const uint16_t*>(p));
}

template <int D>
__device__ __forceinline__ uint32_t fc_pick(const uint4* run, int i0, int i1) {
  const uint32_t* w = reinterpret_cast<const uint32_t*>(run);
  const uint32_t sel = static_cast<uint32_t>((i0 & 1) * 2 | ((i0 & 1) * 2 + 1) << 8 | (4 + (i1 & 1) * 2) << 16 | (4 + (i1 & 1) * 2 + 1) << 24);
  return __builtin_amdgcn_perm(w[i1 >> 1], w[i0 >> 1], sel);
}

// T[i] = source_i W (32 columns from n0) for the DS components of one source block; n: this lane's column, clamped
template <typename TI, int DS, bool WT, bool MI>
__device__ __forceinline__ void fc_products(fx16 (&T)[DS], const FcPart& part, const TI* __restrict__ row, const TI* __restrict__ W, int n) {
  constexpr int ES = sizeof(TI), EPV = 16 / ES, STEP = 2 * EPV;
  const int h = (threadIdx.x >> 5) & 1;
#pragma unroll
  for (int i = 0; i < DS; ++i) T[i] = fx16{0};
  uint4 x[DS], xn[DS], wv, wn;
  auto load = [&](int k0, uint4 (&xx)[DS], uint4& ww) {
    const int k = k0 + EPV * h;
#pragma unroll
    for (int i = 0; i < DS; ++i) xx[i] = *reinterpret_cast<const uint4*>(row + part.a0 + (MI ? k * DS + i * EPV : i * part.K + k));
    if constexpr (WT) {
      ww = *reinterpret_cast<const uint4*>(W + part.w0 + static_cast<int64_t>(n) * part.stride + k);
    } else if constexpr (ES == 4) {
      uint32_t e[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) e[s] = reinterpret_cast<const uint32_t*>(W)[part.w0 + static_cast<int64_t>(k + s) * part.stride + n];
      ww = make_uint4(e[0], e[1], e[2], e[3]);
    } else {
      uint32_t e[8];
#pragma unroll
      for (int s = 0; s < 8; ++s) e[s] = reinterpret_cast<const uint16_t*>(W)[part.w0 + static_cast<int64_t>(k + s) * part.stride + n];
      ww = make_uint4(e[0] | e[1] << 16, e[2] | e[3] << 16, e[4] | e[5] << 16, e[6] | e[7] << 16);
    }
  };
  load(0, x, wv);
  for (int k0 = 0; k0 < part.K; k0 += STEP) {
    load(min(k0 + STEP, part.K - STEP), xn, wn);
    if constexpr (ES == 4) {
      const float* xf = reinterpret_cast<const float*>(&x[0]);
      const float* wf = reinterpret_cast<const float*>(&wv);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < DS; ++i) T[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(wf[s], MI ? xf[s * DS + i] : xf[4 * i + s], T[i], 0, 0, 0);
    } else {
#pragma unroll
      for (int i = 0; i < DS; ++i) {
        uint4 op;
        if constexpr (DS == 1 || !MI) op = x[i];
        else op = make_uint4(fc_pick<DS>(&x[0], i, DS + i), fc_pick<DS>(&x[0], 2 * DS + i, 3 * DS + i), fc_pick<DS>(&x[0], 4 * DS + i, 5 * DS + i),
                             fc_pick<DS>(&x[0], 6 * DS + i, 7 * DS + i));
        T[i] = mm_32x32x16<TI>(wv, op, T[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < DS; ++i) x[i] = xn[i];
    wv = wn;
  }
}

// four adjacent channels m .. m + 3, DR components, of a row of the result side (x1 in the dx2 sums)
template <typename TI, int DR, bool MI>
__device__ __forceinline__ void fc_load4(float (&v)[4][DR], const TI* __restrict__ p, int m, int N) {
#pragma unroll
  for (int q = 0; q < DR; ++q) {
    const TI* src = MI ? p + m * DR + 4 * q : p + q * N + m;
    float f[4];
    if constexpr (sizeof(TI) == 4) {
      const float4 t = *reinterpret_cast<const float4*>(src);
      f[0] = t.x; f[1] = t.y; f[2] = t.z; f[3] = t.w;
    } else {
      const uint2 t = *reinterpret_cast<const uint2*>(src);
      f[0] = mm_widen<TI>(static_cast<uint16_t>(t.x & 0xffff)); f[1] = mm_widen<TI>(static_cast<uint16_t>(t.x >> 16));
      f[2] = mm_widen<TI>(static_cast<uint16_t>(t.y & 0xffff)); f[3] = mm_widen<TI>(static_cast<uint16_t>(t.y >> 16));
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (MI) v[(4 * q + e) / DR][(4 * q + e) % DR] = f[e];
      else v[e][q] = f[e];
    }
  }
}

template <typename TI, int DS, int DR, bool WT, bool MI, bool DX2>
__device__ __forceinline__ void fc_part(fx16 (&acc)[DR], const FcPart& part, const FcBlock& blk, const TI* __restrict__ row, const TI* __restrict__ W,
                                        const float* __restrict__ coef, const TI* __restrict__ x2row, const TI* __restrict__ x1row, float* lsum, int n2, int n0,
                                        int n) {
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  fx16 T[DS];
  fc_products<TI, DS, WT, MI>(T, part, row, W, n);
  const float* __restrict__ cf = coef + part.coef;
  float s[DS][DR];
#pragma unroll
  for (int i = 0; i < DS; ++i)
#pragma unroll
    for (int k = 0; k < DR; ++k) s[i][k] = 0.f;
  for (int j = 0; j < part.d2; ++j) {
    const float xj = fc_widen(x2row + part.j0 + j);
#pragma unroll
    for (int i = 0; i < DS; ++i)
#pragma unroll
      for (int k = 0; k < DR; ++k) s[i][k] = fmaf(cf[(i * DR + k) * part.d2 + j], xj, s[i][k]);
  }
#pragma unroll
  for (int k = 0; k < DR; ++k)
#pragma unroll
    for (int i = 0; i < DS; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[k][v] = fmaf(s[i][k], T[i][v], acc[k][v]);
  if constexpr (DX2) {
    float y[DS][DR];
#pragma unroll
    for (int i = 0; i < DS; ++i)
#pragma unroll
      for (int k = 0; k < DR; ++k) y[i][k] = 0.f;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int m = n0 + 8 * a + 4 * h;
      if (m < blk.N) {
        float xv[4][DR];
        fc_load4<TI, DR, MI>(xv, x1row + blk.c0, m, blk.N);
#pragma unroll
        for (int i = 0; i < DS; ++i)
#pragma unroll
          for (int k = 0; k < DR; ++k)
#pragma unroll
            for (int b = 0; b < 4; ++b) y[i][k] = fmaf(T[i][4 * a + b], xv[b][k], y[i][k]);
      }
    }
#pragma unroll
    for (int i = 0; i < DS; ++i)
#pragma unroll
      for (int k = 0; k < DR; ++k) y[i][k] += __shfl_xor(y[i][k], 32, 64);
    // (the two halves hold the same sums: each takes every other column)
    for (int j = h; j < part.d2; j += 2) {
      float d = 0.f;
#pragma unroll
      for (int i = 0; i < DS; ++i)
#pragma unroll
        for (int k = 0; k < DR; ++k) d = fmaf(cf[(i * DR + k) * part.d2 + j], y[i][k], d);
      lsum[c * n2 + part.j0 + j] += d;
    }
  }
}

template <typename TI, int DR, bool WT, bool MI, bool DX2, int MAXD>
__device__ __forceinline__ void fc_tile(const FcBlock& blk, const FcPart* __restrict__ parts, const float* __restrict__ coef, const TI* __restrict__ A, int64_t lda,
                                        const TI* __restrict__ W, const TI* __restrict__ X2, int64_t ldx2, const TI* __restrict__ X1, int64_t ldx1,
                                        TI* __restrict__ C, int64_t ldc, float* __restrict__ partial, float* lsum, int n2, int64_t Z, int64_t z0, int n0) {
  constexpr int ES = sizeof(TI);
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int64_t z = min(z0 + c, Z - 1);
  fx16 acc[DR];
#pragma unroll
  for (int k = 0; k < DR; ++k) acc[k] = fx16{0};
  if constexpr (DX2) {
    for (int e = lane; e < 32 * n2; e += 64) lsum[e] = 0.f;
    __builtin_amdgcn_wave_barrier();
  }
  const int n = min(n0 + c, blk.N - 1);
  const TI *row = A + z * lda, *x2row = X2 + z * ldx2, *x1row = DX2 ? X1 + z * ldx1 : nullptr;
  for (int p = 0; p < blk.parts; ++p) {
    const FcPart part = parts[blk.first + p];
    switch (part.D) {
      case 1: fc_part<TI, 1, DR, WT, MI, DX2>(acc, part, blk, row, W, coef, x2row, x1row, lsum, n2, n0, n); break;
      case 3: fc_part<TI, 3, DR, WT, MI, DX2>(acc, part, blk, row, W, coef, x2row, x1row, lsum, n2, n0, n); break;
      default:
        if constexpr (MAXD > 3) fc_part<TI, 5, DR, WT, MI, DX2>(acc, part, blk, row, W, coef, x2row, x1row, lsum, n2, n0, n);
    }
  }
  if (z0 + c < Z) {
    TI* out = C + z * ldc + blk.c0;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int m = n0 + 8 * a + 4 * h;
      if (m >= blk.N) continue;
#pragma unroll
      for (int q = 0; q < DR; ++q) {
        float f[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = MI ? acc[(4 * q + e) % DR][4 * a + (4 * q + e) / DR] : acc[q][4 * a + e];
        TI* to = MI ? out + m * DR + 4 * q : out + q * blk.N + m;
        if constexpr (ES == 4) *reinterpret_cast<float4*>(to) = make_float4(f[0], f[1], f[2], f[3]);
        else *reinterpret_cast<uint2*>(to) = make_uint2(mm_pack<TI>(f[0], f[1]), mm_pack<TI>(f[2], f[3]));
      }
    }
  }
  if constexpr (DX2) {
    __builtin_amdgcn_wave_barrier();
    const int64_t rows = min<int64_t>(32, Z - z0);
    for (int e = lane; e < rows * n2; e += 64) partial[z0 * n2 + e] = lsum[e];
  }
}

// MAXD: the most components of any block (3 or 5): what the register budget has to hold
template <typename TI, bool WT, bool MI, bool DX2, int MAXD>
__global__ void __launch_bounds__(256, (MAXD > 3 ? 2 : 3)) fc_rows_kernel(const FcBlock* __restrict__ blocks, const FcPart* __restrict__ parts, const float* __restrict__ coef, int nblocks,
                                                         int tiles_n, const TI* __restrict__ A, int64_t lda, const TI* __restrict__ W, const TI* __restrict__ X2,
                                                         int64_t ldx2, const TI* __restrict__ X1, int64_t ldx1, TI* __restrict__ C, int64_t ldc,
                                                         float* __restrict__ partial, int n2, int64_t Z) {
  extern __shared__ float fc_lsum[];
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int64_t unit = static_cast<int64_t>(blockIdx.x) * 4 + wave;
  const int64_t zt = unit / tiles_n;
  const int column = static_cast<int>(unit - zt * tiles_n);
  int tile = column, b = 0;
  while (b < nblocks && tile >= blocks[b].nt) tile -= blocks[b++].nt;
  const int64_t z0 = zt * 32;
  if (b == nblocks || z0 >= Z) return;
  const FcBlock blk = blocks[b];
  float* lsum = fc_lsum + wave * 32 * n2;
  float* part = DX2 ? partial + static_cast<int64_t>(column) * Z * n2 : nullptr;
  switch (blk.D) {
    case 1: fc_tile<TI, 1, WT, MI, DX2, MAXD>(blk, parts, coef, A, lda, W, X2, ldx2, X1, ldx1, C, ldc, part, lsum, n2, Z, z0, tile * 32); break;
    case 3: fc_tile<TI, 3, WT, MI, DX2, MAXD>(blk, parts, coef, A, lda, W, X2, ldx2, X1, ldx1, C, ldc, part, lsum, n2, Z, z0, tile * 32); break;
    default:
      if constexpr (MAXD > 3) fc_tile<TI, 5, WT, MI, DX2, MAXD>(blk, parts, coef, A, lda, W, X2, ldx2, X1, ldx1, C, ldc, part, lsum, n2, Z, z0, tile * 32);
  }
}

// dx2[z, j] = sum of the partial rows of all column tiles, in order
template <typename TI>
__global__ void __launch_bounds__(256) fc_fold_kernel(const float* __restrict__ partial, TI* __restrict__ out, int64_t values, int tiles) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= values) return;
  float s = 0.f;
  for (int t = 0; t < tiles; ++t) s += partial[t * values + i];
  if constexpr (sizeof(TI) == 4) out[i] = s;
  else reinterpret_cast<uint16_t*>(out)[i] = mm_round<TI>(s);
}

struct FcGrad {  // weight gradient of one path
  int64_t w0;
  int32_t a0, K, D1, c0, N, D3, coef, j0, d2, nt, ntv, unused;
};

template <typename TI, int D1, int D3, bool MI>
__device__ __forceinline__ void fc_grad_tile(const FcGrad& q, int tile, const float* __restrict__ coef, const TI* __restrict__ X1, int64_t ldx1,
                                             const TI* __restrict__ X2, int64_t ldx2, const TI* __restrict__ G, int64_t ldg, float* __restrict__ P, int64_t zb,
                                             int64_t ze) {
  constexpr int ES = sizeof(TI);
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int u0 = (tile / q.ntv) * 64, v0 = (tile % q.ntv) * 64;
  const float* __restrict__ cf = coef + q.coef;
  fx16 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = fx16{0};
  int u[2], v[2];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    u[a] = min(u0 + 32 * a + c, q.K - 1);
    v[a] = min(v0 + 32 * a + c, q.N - 1);
  }
  // x1_i at the lane's two channels and H_i = sum_k s_ik g_k at its two columns, for row z and the components i0 .. i0 + NI (nothing
  // past the chunk)
  auto row_values = [&](int64_t z, int i0, auto ni, float (*x)[decltype(ni)::value], float (*hv)[decltype(ni)::value]) {
    constexpr int NI = decltype(ni)::value;
    const int64_t zr = min(z, ze - 1);
    const bool in = z < ze;
    const TI *xr = X1 + zr * ldx1 + q.a0, *gr = G + zr * ldg + q.c0, *yr = X2 + zr * ldx2 + q.j0;
    float s[NI][D3];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int k = 0; k < D3; ++k) s[i][k] = 0.f;
    for (int j = 0; j < q.d2; ++j) {
      const float xj = fc_widen(yr + j);
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int k = 0; k < D3; ++k) s[i][k] = fmaf(cf[((i0 + i) * D3 + k) * q.d2 + j], xj, s[i][k]);
    }
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      float g[D3];
#pragma unroll
      for (int k = 0; k < D3; ++k) g[k] = fc_widen(gr + (MI ? v[a] * D3 + k : k * q.N + v[a]));
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const float xv = fc_widen(xr + (MI ? u[a] * D1 + i0 + i : (i0 + i) * q.K + u[a]));
        x[a][i] = in ? xv : 0.f;
        float t = 0.f;
#pragma unroll
        for (int k = 0; k < D3; ++k) t = fmaf(s[i][k], g[k], t);
        hv[a][i] = in ? t : 0.f;
      }
    }
  };
  if constexpr (ES == 4) {
    for (int64_t z = zb; z < ze; z += 4) {
      float x[2][2][D1], hv[2][2][D1];
#pragma unroll
      for (int r = 0; r < 2; ++r) row_values(z + 2 * r + h, 0, std::integral_constant<int, D1>{}, x[r], hv[r]);
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int i = 0; i < D1; ++i)
#pragma unroll
          for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[r][a][i], hv[r][b][i], acc[a][b], 0, 0, 0);
    }
  } else {
    for (int64_t z = zb; z < ze; z += 16)
#pragma unroll 1
      for (int i = 0; i < D1; ++i) {  // (a component at a time: eight rows of all of them do not fit the registers)
        uint32_t xp[2][4], hp[2][4];
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          float x[2][2][1], hv[2][2][1];
#pragma unroll
          for (int r = 0; r < 2; ++r) row_values(z + 8 * h + e + r, i, std::integral_constant<int, 1>{}, x[r], hv[r]);
#pragma unroll
          for (int a = 0; a < 2; ++a) {
            xp[a][e >> 1] = mm_pack<TI>(x[0][a][0], x[1][a][0]);
            hp[a][e >> 1] = mm_pack<TI>(hv[0][a][0], hv[1][a][0]);
          }
        }
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b)
            acc[a][b] = mm_32x32x16<TI>(make_uint4(xp[a][0], xp[a][1], xp[a][2], xp[a][3]), make_uint4(hp[b][0], hp[b][1], hp[b][2], hp[b][3]), acc[a][b]);
      }
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int vv = v0 + 32 * b + c;
      if (vv >= q.N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int uu = u0 + 32 * a + 8 * (r >> 2) + 4 * h + (r & 3);
        if (uu < q.K) P[q.w0 + static_cast<int64_t>(uu) * q.N + vv] = acc[a][b][r];
      }
    }
}

template <typename TI, bool MI>
__global__ void __launch_bounds__(256, 2) fc_grad_kernel(const FcGrad* __restrict__ grads, const float* __restrict__ coef, int ngrads, int tiles,
                                                         const TI* __restrict__ X1, int64_t ldx1, const TI* __restrict__ X2, int64_t ldx2, const TI* __restrict__ G,
                                                         int64_t ldg, float* __restrict__ partial, int64_t numel, int64_t Z, int64_t rows_per_chunk, int64_t chunks) {
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int64_t unit = static_cast<int64_t>(blockIdx.x) * 4 + wave;
  const int64_t chunk = unit / tiles;
  if (chunk >= chunks) return;
  int tile = static_cast<int>(unit - chunk * tiles), b = 0;
  while (b < ngrads && tile >= grads[b].nt) tile -= grads[b++].nt;
  if (b == ngrads) return;
  const FcGrad q = grads[b];
  const int64_t zb = chunk * rows_per_chunk, ze = min(zb + rows_per_chunk, Z);
  float* P = partial + chunk * numel;
#define FC_TILE(A, B) fc_grad_tile<TI, A, B, MI>(q, tile, coef, X1, ldx1, X2, ldx2, G, ldg, P, zb, ze)
  switch (q.D1 * 8 + q.D3) {
    case 9: FC_TILE(1, 1); break;
    case 11: FC_TILE(1, 3); break;
    case 13: FC_TILE(1, 5); break;
    case 25: FC_TILE(3, 1); break;
    case 27: FC_TILE(3, 3); break;
    case 29: FC_TILE(3, 5); break;
    case 41: FC_TILE(5, 1); break;
    case 43: FC_TILE(5, 3); break;
    default: FC_TILE(5, 5);
  }
#undef FC_TILE
}

// H_p,i = sum_k s_ik g_k for all rows, written out (columns path after path, component after component), and x1 with its
// components apart where it is stored mul_ir: what the weight gradient contracts as plain products once there are rows enough
// for the tiled kernel (above, every 64 x 64 tile forms its H again: 395 us for 128 channels and 50 000 rows of bfloat16, 128 so).
template <typename TI, bool MI>
__global__ void __launch_bounds__(256) fc_factors_kernel(const FcGrad* __restrict__ grads, const float* __restrict__ coef, int ngrads,
                                                         const FcBlock* __restrict__ blocks1, int nblocks1, const TI* __restrict__ X1, int64_t ldx1,
                                                         const TI* __restrict__ X2, int64_t ldx2, const TI* __restrict__ G, int64_t ldg, TI* __restrict__ H,
                                                         int64_t ldh, TI* __restrict__ X1T, int64_t Z, int nfactors) {
  extern __shared__ float fc_lfac[];  // (a row of factors per wavefront)
  const int lane = threadIdx.x & 63;
  float* s = fc_lfac + (threadIdx.x >> 6) * nfactors;
  auto store2 = [&](TI* to, float a, float b) {
    if constexpr (sizeof(TI) == 4) *reinterpret_cast<float2*>(to) = make_float2(a, b);
    else *reinterpret_cast<uint32_t*>(to) = mm_pack<TI>(a, b);
  };
  for (int64_t z = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6); z < Z; z += static_cast<int64_t>(gridDim.x) * 4) {
    TI* h = H + z * ldh;
    int off = 0;
    __builtin_amdgcn_wave_barrier();
    for (int p = 0; p < ngrads; ++p) {  // the factors of the row, a lane each
      const FcGrad q = grads[p];
      const TI* yr = X2 + z * ldx2 + q.j0;
      const int n = q.D1 * q.D3;
      if (lane < n) {
        float f = 0.f;
        for (int j = 0; j < q.d2; ++j) f = fmaf(coef[q.coef + lane * q.d2 + j], fc_widen(yr + j), f);
        s[off + lane] = f;
      }
      off += n;
    }
    __builtin_amdgcn_wave_barrier();
    off = 0;
    for (int p = 0; p < ngrads; ++p) {
      const FcGrad q = grads[p];
      const TI* gr = G + z * ldg + q.c0;
      for (int w = 2 * lane; w < q.N; w += 128) {
        float ga[5], gb[5];
#pragma unroll
        for (int k = 0; k < 5; ++k)
          if (k < q.D3) {
            ga[k] = fc_widen(gr + (MI ? w * q.D3 + k : k * q.N + w));
            gb[k] = fc_widen(gr + (MI ? (w + 1) * q.D3 + k : k * q.N + w + 1));
          }
        for (int i = 0; i < q.D1; ++i) {
          float a = 0.f, b = 0.f;
#pragma unroll
          for (int k = 0; k < 5; ++k)
            if (k < q.D3) {
              const float f = s[off + i * q.D3 + k];
              a = fmaf(f, ga[k], a);
              b = fmaf(f, gb[k], b);
            }
          store2(h + i * q.N + w, a, b);
        }
      }
      h += q.D1 * q.N;
      off += q.D1 * q.D3;
    }
    if constexpr (MI) {
      for (int b = 0; b < nblocks1; ++b) {
        const FcBlock blk = blocks1[b];
        const TI* src = X1 + z * ldx1 + blk.c0;
        TI* dst = X1T + z * ldx1 + blk.c0;
        for (int u = 2 * lane; u < blk.N; u += 128)
          for (int i = 0; i < blk.D; ++i) store2(dst + i * blk.N + u, fc_widen(src + u * blk.D + i), fc_widen(src + (u + 1) * blk.D + i));
      }
    }
  }
}

}  // namespace
}  // namespace cueq

using namespace cueq;

static_assert(sizeof(FcPart) == 40 && sizeof(FcBlock) == 24 && sizeof(FcGrad) == 56, "the tables the host uploads");

#define FC_DISPATCH(dt, CALL)                                      \
  do {                                                             \
    if ((dt) == CUEQ_F32) { CALL(float); }                         \
    else if ((dt) == CUEQ_F16) { CALL(f16bits); }                  \
    else { CALL(uint16_t); }                                       \
  } while (0)

// gradient == 0: rows of x1 against W; 1: rows of the cotangent against W^T, and with X1, partial and dX2 given also the gradient of x2
extern "C" int cueq_fc_flex(int32_t dtype, int32_t gradient, int32_t mul_ir, int64_t rows, const void* A, int64_t lda, const void* W, const void* X2, int64_t ldx2,
                            const void* X1, int64_t ldx1, void* C, int64_t ldc, const void* blocks, int32_t nblocks, const void* parts, const float* coef,
                            int32_t column_tiles, int32_t most_components, int32_t n2, float* partial, void* dX2, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  CUEQ_REQUIRE(dtype == CUEQ_F32 || dtype == CUEQ_BF16 || dtype == CUEQ_F16, CUEQ_ERR_UNSUPPORTED, "fc_flex: dtype must be float32, bfloat16 or half");
  CUEQ_REQUIRE(rows >= 0 && nblocks > 0 && column_tiles > 0 && n2 > 0 && n2 <= 64, CUEQ_ERR_INVALID, "fc_flex: bad extents");
  if (rows == 0) return CUEQ_OK;
  CUEQ_REQUIRE(A && W && X2 && C && blocks && parts && coef && (!dX2 || (gradient && X1 && partial)), CUEQ_ERR_INVALID, "fc_flex: null operand");
  const int64_t epv = dtype == CUEQ_F32 ? 4 : 8;
  CUEQ_REQUIRE(((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(C) | reinterpret_cast<uintptr_t>(W) | reinterpret_cast<uintptr_t>(X1)) & 15) == 0 &&
                   lda % epv == 0 && ldc % epv == 0 && ldx1 % epv == 0,
               CUEQ_ERR_UNSUPPORTED, "fc_flex: rows must be 16-byte aligned");
  const int64_t units = (rows + 31) / 32 * column_tiles, grid = (units + 3) / 4;
  CUEQ_REQUIRE(grid < (1ll << 31), CUEQ_ERR_TOO_LARGE, "fc_flex: too many rows");
  const size_t lds = dX2 ? 4 * 32 * n2 * sizeof(float) : 0;
  KernelTimer timer(gradient ? "fc_flex_dx" : "fc_flex_fwd", stream);
#define FC_GO(TI, WT, MI, DX) do { if (most_components <= 3) FC_GD(TI, WT, MI, DX, 3); else FC_GD(TI, WT, MI, DX, 5); } while (0)
#define FC_GD(TI, WT, MI, DX, MD) hipLaunchKernelGGL((fc_rows_kernel<TI, WT, MI, DX, MD>), dim3(static_cast<unsigned>(grid)), dim3(256), lds, stream, static_cast<const FcBlock*>(blocks), static_cast<const FcPart*>(parts), coef, nblocks, column_tiles, static_cast<const TI*>(A), lda, static_cast<const TI*>(W), static_cast<const TI*>(X2), ldx2, static_cast<const TI*>(X1), ldx1, static_cast<TI*>(C), ldc, partial, n2, rows)
#define FC(TI)                                                                                     \
  do {                                                                                             \
    if (!gradient) { if (mul_ir) FC_GO(TI, false, true, false); else FC_GO(TI, false, false, false); } \
    else if (dX2) { if (mul_ir) FC_GO(TI, true, true, true); else FC_GO(TI, true, false, true); }  \
    else { if (mul_ir) FC_GO(TI, true, true, false); else FC_GO(TI, true, false, false); }         \
  } while (0)
  FC_DISPATCH(dtype, FC);
#undef FC
#undef FC_GD
#undef FC_GO
  CUEQ_CHECK_HIP(hipGetLastError());
  if (dX2) {
    const int64_t values = rows * n2;
#define FC(TI) hipLaunchKernelGGL(fc_fold_kernel<TI>, dim3(static_cast<unsigned>((values + 255) / 256)), dim3(256), 0, stream, partial, static_cast<TI*>(dX2), values, column_tiles)
    FC_DISPATCH(dtype, FC);
#undef FC
    CUEQ_CHECK_HIP(hipGetLastError());
  }
  return CUEQ_OK;
}

// partial products of every path's weight gradient: cueq_fc_flex_dw_chunks x numel floats, to be summed in order (cueq_sum_runs)
static int64_t fc_rows_per_chunk(int64_t rows, int32_t tiles) {
  int64_t chunks = std::min<int64_t>(8ll * device_cus() / std::max(1, tiles), (rows + 15) / 16);
  chunks = std::max<int64_t>(1, chunks);
  return ((rows + chunks - 1) / chunks + 15) / 16 * 16;
}
extern "C" int64_t cueq_fc_flex_dw_chunks(int64_t rows, int32_t tiles) {
  const int64_t rpc = fc_rows_per_chunk(rows, tiles);
  return (rows + rpc - 1) / rpc;
}
extern "C" int cueq_fc_flex_dw(int32_t dtype, int32_t mul_ir, int64_t rows, const void* X1, int64_t ldx1, const void* X2, int64_t ldx2, const void* G, int64_t ldg,
                               const void* grads, int32_t ngrads, const float* coef, int32_t tiles, int64_t numel, float* partial, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  CUEQ_REQUIRE(dtype == CUEQ_F32 || dtype == CUEQ_BF16 || dtype == CUEQ_F16, CUEQ_ERR_UNSUPPORTED, "fc_flex_dw: dtype must be float32, bfloat16 or half");
  CUEQ_REQUIRE(rows > 0 && ngrads > 0 && tiles > 0 && numel > 0, CUEQ_ERR_INVALID, "fc_flex_dw: bad extents");
  CUEQ_REQUIRE(X1 && X2 && G && grads && coef && partial, CUEQ_ERR_INVALID, "fc_flex_dw: null operand");
  const int64_t rpc = fc_rows_per_chunk(rows, tiles), chunks = (rows + rpc - 1) / rpc, grid = (chunks * tiles + 3) / 4;
  CUEQ_REQUIRE(grid < (1ll << 31), CUEQ_ERR_TOO_LARGE, "fc_flex_dw: too many tiles");
  KernelTimer timer("fc_flex_dw", stream);
#define FC_GO(TI, MI) hipLaunchKernelGGL((fc_grad_kernel<TI, MI>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, static_cast<const FcGrad*>(grads), coef, ngrads, tiles, static_cast<const TI*>(X1), ldx1, static_cast<const TI*>(X2), ldx2, static_cast<const TI*>(G), ldg, partial, numel, rows, rpc, chunks)
#define FC(TI) do { if (mul_ir) FC_GO(TI, true); else FC_GO(TI, false); } while (0)
  FC_DISPATCH(dtype, FC);
#undef FC
#undef FC_GO
  CUEQ_CHECK_HIP(hipGetLastError());
  return CUEQ_OK;
}

extern "C" int cueq_fc_factors(int32_t dtype, int32_t mul_ir, int64_t rows, const void* X1, int64_t ldx1, const void* X2, int64_t ldx2, const void* G, int64_t ldg,
                               const void* grads, int32_t ngrads, const float* coef, const void* blocks1, int32_t nblocks1, int32_t nfactors, void* H, int64_t ldh, void* X1T,
                               void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  CUEQ_REQUIRE(dtype == CUEQ_F32 || dtype == CUEQ_BF16 || dtype == CUEQ_F16, CUEQ_ERR_UNSUPPORTED, "fc_factors: dtype must be float32, bfloat16 or half");
  CUEQ_REQUIRE(rows > 0 && X1 && X2 && G && grads && coef && H && (!mul_ir || (X1T && blocks1)), CUEQ_ERR_INVALID, "fc_factors: null operand");
  CUEQ_REQUIRE(nfactors > 0 && nfactors <= 2048, CUEQ_ERR_UNSUPPORTED, "fc_factors: too many factors a row");
  const dim3 grid(static_cast<unsigned>(std::min<int64_t>((rows + 3) / 4, 8ll * device_cus())));
  const size_t lds = 4 * nfactors * sizeof(float);
  KernelTimer timer("fc_factors", stream);
#define FC_GO(TI, MI) hipLaunchKernelGGL((fc_factors_kernel<TI, MI>), grid, dim3(256), lds, stream, static_cast<const FcGrad*>(grads), coef, ngrads, static_cast<const FcBlock*>(blocks1), nblocks1, static_cast<const TI*>(X1), ldx1, static_cast<const TI*>(X2), ldx2, static_cast<const TI*>(G), ldg, static_cast<TI*>(H), ldh, static_cast<TI*>(X1T), rows, nfactors)
#define FC(TI) do { if (mul_ir) FC_GO(TI, true); else FC_GO(TI, false); } while (0)
  FC_DISPATCH(dtype, FC);
#undef FC
#undef FC_GO
  CUEQ_CHECK_HIP(hipGetLastError());
  return CUEQ_OK;
}
