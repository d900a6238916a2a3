// Fully connected product with shared weights (uvw,iu,jv,kw+ijk, any v), table-driven:
//
//   out[z, k, w] = sum over the paths p of the block and the channels v of its x2 block
//                  sum_ij C_p[i, j, k] x2[z, j, v] sum_u x1[z, i, u] W_p[u, v, w]
//
// First for one channel v (a second operand of multiplicity one, and float rows of any): a channel is a part of its own.
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

struct FcPart {            // one path: its weights, the source block it contracts, its factors
  int64_t w0;
  int32_t a0, K, D, coef;  // source block: offset, multiplicity, components; coef: offset of the D x DR x d2 factors
  int32_t j0, d2;          // x2 block: offset, components
  int32_t stride, V, js, vs, wv;  // elements between weight rows as stored; multiplicity of the x2 block, elements between its
                                  // components / its channels, and between the weights of two channels
  uint32_t mask;           // bit i * DR + k: some factor of (i, k) is not zero
};
struct FcPack {  // the weights of one path put into the order of the matrix instructions' operands
  int64_t src, dst;
  int32_t K, N, sk, sn, V, vs, pieces, steps;  // contracted / result extent and their strides, channels of x2 and their stride;
                                               // steps of 16 contracted values written (zeros past K)
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

// component i of eight channels: x is DS pieces of one component each (ir_mul) or of eight channels with their components adjacent
template <int DS, bool MI>
__device__ __forceinline__ uint4 fc_component(const uint4 (&x)[DS], int i) {
  if constexpr (DS == 1 || !MI) return x[i];
  else return make_uint4(mm_pick(&x[0], i, DS + i), mm_pick(&x[0], 2 * DS + i, 3 * DS + i), mm_pick(&x[0], 4 * DS + i, 5 * DS + i),
                         mm_pick(&x[0], 6 * DS + i, 7 * DS + i));
}

// The coefficients of one path (at most 64), a lane each: short products would wait for a memory request for each of them.
struct FcCoefs {
  float mine;
  __device__ __forceinline__ FcCoefs(const float* from, int n) : mine(0.f) {
    const int lane = threadIdx.x & 63;
    if (lane < n) mine = from[lane];
  }
  __device__ __forceinline__ float operator[](int i) const {  // i: the same in all lanes
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mine), i));
  }
};

// How the weights lie: as given, contracted over their first or their last extent, or packed by fc_pack_kernel
enum FcWeights { kPlain = 0, kTransposed = 1, kPacked = 2 };
constexpr int kFragment = 512;  // 2-byte elements of one packed operand: 64 lanes x 8

// T[i] = source_i W (32 columns from n0) for the DS components of one source block; n: this lane's column, clamped; W: the weights of
// the path and the channel of x2
template <typename TI, int DS, int WM, bool MI>
__device__ __forceinline__ void fc_products(fx16 (&T)[DS], const FcPart& part, const TI* __restrict__ row, const TI* __restrict__ W, int n, int n0) {
  constexpr int ES = sizeof(TI), EPV = 16 / ES, STEP = 2 * EPV;
  const int h = (threadIdx.x >> 5) & 1;
#pragma unroll
  for (int i = 0; i < DS; ++i) T[i] = fx16{0};
  uint4 x[DS], xn[DS], wv, wn;
  auto load = [&](int k0, uint4 (&xx)[DS], uint4& ww) {
    const int k = k0 + EPV * h;
#pragma unroll
    for (int i = 0; i < DS; ++i) xx[i] = *reinterpret_cast<const uint4*>(row + part.a0 + (MI ? k * DS + i * EPV : i * part.K + k));
    if constexpr (WM == kPacked) {
      ww = *reinterpret_cast<const uint4*>(W + ((k0 / STEP) * part.stride + n0 / 32) * kFragment + (threadIdx.x & 63) * 8);
    } else if constexpr (WM == kTransposed) {
      ww = *reinterpret_cast<const uint4*>(W + static_cast<int64_t>(n) * part.stride + k);
    } else if constexpr (ES == 4) {
      uint32_t e[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) e[s] = reinterpret_cast<const uint32_t*>(W)[static_cast<int64_t>(k + s) * part.stride + n];
      ww = make_uint4(e[0], e[1], e[2], e[3]);
    } else {
      uint32_t e[8];
#pragma unroll
      for (int s = 0; s < 8; ++s) e[s] = reinterpret_cast<const uint16_t*>(W)[static_cast<int64_t>(k + s) * part.stride + n];
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
        T[i] = mm_32x32x16<TI>(wv, fc_component<DS, MI>(x, i), T[i]);
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

// Structural zeros.  The plain kernels multiply every pair of components by its factor, those that no coefficient couples among
// them: with finite values a factor of zero adds nothing, but 0 * inf would make the whole row NaN where one component has
// overflowed.  Results that are all finite have met finite values only; a wavefront that finds one of its results infinite or undefined
// leaves the tile to fc_tile_coupled / fc_grad_coupled, which touch coupled components alone, in a simple loop of few registers
// behind the straight code.  Tests for couplings in the straight code instead: forward of 3 000 rows of
// 64 channels up to l = 2 (x) 8, float, 234 -> 280 us.
__device__ __forceinline__ float fc_coupled(float c, float x, float s) { return fmaf(c, c == 0.f ? 0.f : x, s); }
__device__ __forceinline__ float fc_probe(const fx16& v, float probe) {  // stays 0 while everything is finite
#pragma unroll
  for (int r = 0; r < 16; ++r) probe = fmaf(v[r], 0.f, probe);
  return probe;
}

// one tile: a row and half of the columns a lane, four at a time; with X1 also the row sums of the gradient of x2
template <typename TI>
__device__ __forceinline__ void fc_tile_coupled(const FcBlock* __restrict__ block, const FcPart* __restrict__ parts, const float* __restrict__ coef,
                                                          const TI* __restrict__ A, int64_t lda, const TI* __restrict__ W, const TI* __restrict__ X2,
                                                          int64_t ldx2, const TI* __restrict__ X1, int64_t ldx1, TI* __restrict__ C, int64_t ldc,
                                                          float* __restrict__ partial, float* lsum, int wm, bool mi, int n2, int64_t Z, int64_t z0, int n0) {
  const FcBlock blk = *block;
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5, DR = blk.D, n2p = n2 | 1;
  const int64_t z = min(z0 + c, Z - 1);
  const TI *row = A + z * lda, *x2row = X2 + z * ldx2, *x1row = X1 ? X1 + z * ldx1 : nullptr;
  float* sums = lsum + c * n2p;
  if (x1row && h == 0)
    for (int j = 0; j < n2; ++j) sums[j] = 0.f;
  __builtin_amdgcn_wave_barrier();
#pragma unroll 1
  for (int m0 = n0 + 16 * h; m0 < n0 + 16 * h + 16; m0 += 4) {
    float acc[5][4];
#pragma unroll
    for (int k = 0; k < 5; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[k][e] = 0.f;
#pragma unroll 1
    for (int p = 0; p < blk.parts; ++p) {
      const FcPart part = parts[blk.first + p];
#pragma unroll 1
      for (int i = 0; i < part.D; ++i) {
        float t[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int u = 0; u < part.K; ++u) {
          const float x = fc_widen(row + part.a0 + (mi ? u * part.D + i : i * part.K + u));
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int n = min(m0 + e, blk.N - 1);
            const int64_t at = wm == kPacked ? static_cast<int64_t>((u >> 4) * part.stride + (n >> 5)) * kFragment + ((u >> 3 & 1) * 32 + (n & 31)) * 8 + (u & 7)
                               : wm == kTransposed ? static_cast<int64_t>(n) * part.stride + u : static_cast<int64_t>(u) * part.stride + n;
            t[e] = fmaf(x, fc_widen(W + part.w0 + at), t[e]);
          }
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) {
          if (k >= DR || !(part.mask >> (i * DR + k) & 1)) continue;
          const float* cf = coef + part.coef + (i * DR + k) * part.d2;
          float s = 0.f;
#pragma unroll 1
          for (int j = 0; j < part.d2; ++j) s = fc_coupled(cf[j], fc_widen(x2row + part.j0 + j * part.js), s);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[k][e] = fmaf(s, t[e], acc[k][e]);
          if (!x1row) continue;
          float y = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (m0 + e < blk.N) y = fmaf(t[e], fc_widen(x1row + blk.c0 + (mi ? (m0 + e) * DR + k : k * blk.N + m0 + e)), y);
          y += __shfl_xor(y, 32, 64);
          if (h == 0)
#pragma unroll 1
            for (int j = 0; j < part.d2; ++j) sums[part.j0 + j * part.js] = fc_coupled(cf[j], y, sums[part.j0 + j * part.js]);
        }
      }
    }
    if (z0 + c >= Z) continue;
    TI* out = C + z * ldc + blk.c0;
#pragma unroll
    for (int k = 0; k < 5; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (k >= DR || m0 + e >= blk.N) continue;
        TI* to = out + (mi ? (m0 + e) * DR + k : k * blk.N + m0 + e);
        if constexpr (sizeof(TI) == 4) *to = acc[k][e];
        else *reinterpret_cast<uint16_t*>(to) = mm_round<TI>(acc[k][e]);
      }
  }
  if (x1row) {
    __builtin_amdgcn_wave_barrier();
    const int64_t rows = min<int64_t>(32, Z - z0);
    for (int e = lane; e < rows * n2; e += 64) partial[z0 * n2 + e] = lsum[e / n2 * n2p + e % n2];
  }
}

// (a channel of x2 is a part of its own here: a loop over them costs the registers of straight code)
template <typename TI, int DS, int DR, int WM, bool MI, bool DX2>
__device__ __forceinline__ void fc_part(fx16 (&acc)[DR], const FcPart& part, const FcBlock& blk, const TI* __restrict__ row, const TI* __restrict__ W,
                                        const float* __restrict__ coef, const TI* __restrict__ x2row, const TI* __restrict__ x1row, float* sums, int n0, int n) {
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const float* __restrict__ cf = coef + part.coef;
  fx16 T[DS];
  fc_products<TI, DS, WM, MI>(T, part, row, W + part.w0, n, n0);
  float s[DS][DR];
#pragma unroll
  for (int i = 0; i < DS; ++i)
#pragma unroll
    for (int k = 0; k < DR; ++k) s[i][k] = 0.f;
  for (int j = 0; j < part.d2; ++j) {
    const float xj = fc_widen(x2row + part.j0 + j * part.js);
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
      for (int r = 0; r < 16; ++r) acc[k][r] = fmaf(s[i][k], T[i][r], acc[k][r]);
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
      sums[part.j0 + j * part.js] += d;
    }
  }
}

// The components that a product of irreps of degree 0 and 1 couples (d1 x d2 -> d3 with d <= 3, and 3 x 5 -> 3, symmetric in the
// two threes): which (i, j, k) have a coefficient at all is known when the kernel is compiled, and its loops are straight code
// that touches nothing else.  The host tests its coefficients against the same rule (_couples in dense.py).
template <int DS, int DR, int D2>
constexpr bool fc_couples(int i, int k, int j) {
  if (DS == 1 && DR == 1) return true;
  if (DS == 1) return j == k;
  if (DR == 1) return j == i;
  if (D2 == 1) return i == k;
  if (D2 == 3) return i != k && j == 3 - i - k;
  return j == 0 ? i + k == 2 && i != k : j == 1 ? i + k == 1 : j == 2 ? i == k : j == 3 ? i + k == 3 : i == k && i != 1;
}
template <int DS, int DR, int D2>
constexpr bool fc_couples(int i, int k) {
  for (int j = 0; j < D2; ++j)
    if (fc_couples<DS, DR, D2>(i, k, j)) return true;
  return false;
}

// 2-byte elements where x2 has several channels, packed weights, K <= 16 KT and the couplings above: the source block of the row stays in registers over
// the channels of x2, and the weights of 16 / KT channels go through LDS for the four wavefronts of the workgroup (four row tiles under
// one column tile), the next ones requested meanwhile.  Straight code is what counts: with the extents, the components of x2 and the
// couplings tested in the loop, every fragment was waited for by itself and a channel took some 3 000 cycles of latency.
// Bound by the issue of vector instructions (a product of 32 x 32 x K is scaled and added component by component); 12 501 rows of
// 64x0e+64x1o (x) 16x0e+16x1o, bfloat16: forward 38.7 us, both input gradients 82 us (the tests in the loop: 45 / 172, x2 read from
// memory: 46), where the products of the operands went through memory 160 and 340 us.
// SK > 1 (few row tiles): the SK wavefronts of the workgroup share one row tile, each with every SK-th channel, its weights from memory.
template <typename TI, int DS, int DR, int D2, bool MI, bool DX2, int KT, int SK>
__device__ __forceinline__ void fc_part_channels(fx16 (&acc)[DR], const FcPart& part, const FcBlock& blk, const TI* __restrict__ row, const TI* __restrict__ W,
                                                 const float* __restrict__ coef, const TI* x2row, const TI* __restrict__ x1row, float* sums, uint4* wl,
                                                 int n0) {
  constexpr int VC = 16 / KT, WN = SK > 1 ? KT : 4;
  const int lane = threadIdx.x & 63, h = lane >> 5, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  if (SK > 1 && wave >= part.V) return;
  uint4 x[KT][DS], wn[WN];
  auto request = [&](int v0) {  // (fragments past K are packed as zeros; past the last channel the last one is read again)
#pragma unroll
    for (int e = 0; e < WN; ++e) {
      const int f = SK > 1 ? e : wave + 4 * e, v = min(v0 + f / KT, part.V - 1), t = f % KT;
      wn[e] = *reinterpret_cast<const uint4*>(W + part.w0 + static_cast<int64_t>(v) * part.wv + (t * part.stride + n0 / 32) * kFragment + lane * 8);
    }
  };
  request(SK > 1 ? wave : 0);
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    const int k = 16 * t + 8 * h, kk = min(k, part.K - 8);
    uint4 raw[DS];
#pragma unroll
    for (int i = 0; i < DS; ++i) raw[i] = *reinterpret_cast<const uint4*>(row + part.a0 + (MI ? kk * DS + i * 8 : i * part.K + kk));
#pragma unroll
    for (int i = 0; i < DS; ++i) x[t][i] = k < part.K ? fc_component<DS, MI>(raw, i) : make_uint4(0, 0, 0, 0);
  }
  uint2 x1[DX2 ? 4 : 1][DR];
  if constexpr (DX2) {
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int m = min(n0 + 8 * a + 4 * h, blk.N - 4);
#pragma unroll
      for (int q = 0; q < DR; ++q) x1[a][q] = *reinterpret_cast<const uint2*>(x1row + blk.c0 + (MI ? m * DR + 4 * q : q * blk.N + m));
    }
  }
  const FcCoefs cf(coef + part.coef, DS * DR * D2);
#pragma unroll 1
  for (int v0 = SK > 1 ? wave : 0; v0 < part.V; v0 += SK > 1 ? SK : VC) {
    uint4 wv[KT];
    if constexpr (SK > 1) {
#pragma unroll
      for (int t = 0; t < KT; ++t) wv[t] = wn[t];
    } else {
      __syncthreads();
#pragma unroll
      for (int e = 0; e < 4; ++e) wl[(wave + 4 * e) * 64 + lane] = wn[e];
      __syncthreads();
    }
    request(v0 + (SK > 1 ? SK : VC));
    const int end = SK > 1 ? 1 : min(VC, part.V - v0);
#pragma unroll 1
    for (int g = 0; g < end; ++g) {
      const int y0 = part.j0 + (v0 + g) * part.vs;
      float xj[D2];
#pragma unroll
      for (int j = 0; j < D2; ++j) xj[j] = fc_widen(x2row + y0 + j * part.js);
      if constexpr (SK == 1)
#pragma unroll
        for (int t = 0; t < KT; ++t) wv[t] = wl[(g * KT + t) * 64 + lane];
      fx16 T[DS];
#pragma unroll
      for (int i = 0; i < DS; ++i) T[i] = fx16{0};
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int i = 0; i < DS; ++i) T[i] = mm_32x32x16<TI>(wv[t], x[t][i], T[i]);
      float s[DS][DR];
#pragma unroll
      for (int i = 0; i < DS; ++i)
#pragma unroll
        for (int k = 0; k < DR; ++k) {
          s[i][k] = 0.f;
          if (fc_couples<DS, DR, D2>(i, k))
#pragma unroll
            for (int j = 0; j < D2; ++j)
              if (fc_couples<DS, DR, D2>(i, k, j)) s[i][k] = fmaf(cf[(i * DR + k) * D2 + j], xj[j], s[i][k]);
        }
#pragma unroll
      for (int k = 0; k < DR; ++k)
#pragma unroll
        for (int i = 0; i < DS; ++i)
          if (fc_couples<DS, DR, D2>(i, k))
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[k][r] = fmaf(s[i][k], T[i][r], acc[k][r]);
      if constexpr (DX2) {
        float y[DS][DR];
#pragma unroll
        for (int i = 0; i < DS; ++i)
#pragma unroll
          for (int k = 0; k < DR; ++k) y[i][k] = 0.f;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const bool in = n0 + 8 * a + 4 * h < blk.N;
          float xv[4][DR];
#pragma unroll
          for (int q = 0; q < DR; ++q) {
            uint32_t w[2] = {x1[a][q].x, x1[a][q].y};
            asm volatile("" : "+v"(w[0]), "+v"(w[1]));  // (widened here, not kept widened over the channels: 48 registers)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float f = mm_widen<TI>(static_cast<uint16_t>(e & 1 ? w[e >> 1] >> 16 : w[e >> 1] & 0xffffu));
              if constexpr (MI) xv[(4 * q + e) / DR][(4 * q + e) % DR] = f;
              else xv[e][q] = f;
            }
          }
#pragma unroll
          for (int i = 0; i < DS; ++i)
#pragma unroll
            for (int k = 0; k < DR; ++k)
              if (fc_couples<DS, DR, D2>(i, k)) {
                float f = 0.f;
#pragma unroll
                for (int b = 0; b < 4; ++b) f = fmaf(T[i][4 * a + b], xv[b][k], f);
                y[i][k] += in ? f : 0.f;
              }
        }
#pragma unroll
        for (int i = 0; i < DS; ++i)
#pragma unroll
          for (int k = 0; k < DR; ++k)
            if (fc_couples<DS, DR, D2>(i, k)) y[i][k] += __shfl_xor(y[i][k], 32, 64);
        // (the two halves hold the same sums: each adds every other column)
#pragma unroll
        for (int j = 0; j < D2; ++j) {
          float d = 0.f;
#pragma unroll
          for (int i = 0; i < DS; ++i)
#pragma unroll
            for (int k = 0; k < DR; ++k)
              if (fc_couples<DS, DR, D2>(i, k, j)) d = fmaf(cf[(i * DR + k) * D2 + j], y[i][k], d);
          if ((j & 1) == h) sums[y0 + j * part.js] += d;
        }
      }
    }
  }
}

// 32-bit words from row to row of x2 in LDS
__host__ __device__ constexpr int fc_x2_words(int n2) { return (n2 + 1) / 2 | 1; }

// false: some result is not finite, nothing is stored.  SK > 1: the SK wavefronts of the workgroup share the tile, each with some of the
// parts (or channels) of its sums; their sums are added in order, and each of the first four stores eight of the columns.
template <typename TI, int DR, int WM, bool MI, bool DX2, int MAXD, int KT, int SK>
__device__ __forceinline__ bool fc_tile(const FcBlock& blk, const FcPart* __restrict__ parts, const float* __restrict__ coef, const TI* __restrict__ A, int64_t lda,
                                        const TI* __restrict__ W, const TI* __restrict__ X2, int64_t ldx2, const TI* __restrict__ X1, int64_t ldx1,
                                        TI* __restrict__ C, int64_t ldc, float* __restrict__ partial, float* lsum, uint4* wl, int n2, int64_t Z, int64_t z0, int n0) {
  constexpr int ES = sizeof(TI);
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int64_t z = min(z0 + c, Z - 1);
  fx16 acc[DR];
#pragma unroll
  for (int k = 0; k < DR; ++k) acc[k] = fx16{0};
  const int n2p = n2 | 1;  // (sums of the lanes' rows an odd number of words apart)
  if constexpr (DX2) {
    for (int e = lane; e < 32 * n2p; e += 64) lsum[e] = 0.f;
    __builtin_amdgcn_wave_barrier();
  }
  const int n = min(n0 + c, blk.N - 1);
  const TI *row = A + z * lda, *x2row = X2 + z * ldx2, *x1row = DX2 ? X1 + z * ldx1 : nullptr;
  if constexpr (KT > 0) {  // the rows of x2 are read channel by channel: from LDS, an odd number of words apart
    const int words = fc_x2_words(n2);
    uint32_t* x2l = reinterpret_cast<uint32_t*>(wl + 16 * 64) + (DX2 ? 4 * 32 * n2p : 0) + (threadIdx.x >> 6) * 32 * words;
    static_assert(KT == 0 || SK == 1 || SK == 4, "four wavefronts' regions of LDS");
    const int used = (n2 + 1) / 2;
#pragma unroll 8
    for (int e = lane; e < 32 * used; e += 64) {
      const int r = e / used, j = 2 * (e - r * used);
      const uint16_t* from = reinterpret_cast<const uint16_t*>(X2 + min(z0 + r, Z - 1) * ldx2 + j);
      x2l[r * words + e - r * used] = static_cast<uint32_t>(from[0]) | static_cast<uint32_t>(from[j + 1 < n2 ? 1 : 0]) << 16;
    }
    __builtin_amdgcn_wave_barrier();
    x2row = reinterpret_cast<const TI*>(x2l + c * words);
  }
  float* sums = lsum + c * n2p;
  auto one = [&](auto ds, const FcPart& part) {
    constexpr int DS = decltype(ds)::value;
    auto channels = [&](auto d2) { fc_part_channels<TI, DS, DR, decltype(d2)::value, MI, DX2, KT, SK>(acc, part, blk, row, W, coef, x2row, x1row, sums, wl, n0); };
    if constexpr (KT > 0 && DS == 3 && DR == 3) {
      if (part.d2 == 1) channels(std::integral_constant<int, 1>{});
      else if (part.d2 == 3) channels(std::integral_constant<int, 3>{});
      else channels(std::integral_constant<int, 5>{});
    } else if constexpr (KT > 0) {
      channels(std::integral_constant<int, (DS == 1 && DR == 1 ? 1 : 3)>{});
    } else {
      fc_part<TI, DS, DR, WM, MI, DX2>(acc, part, blk, row, W, coef, x2row, x1row, sums, n0, n);
    }
  };
  const int share = SK > 1 ? __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)) : 0;
  for (int p = KT == 0 ? share : 0; p < blk.parts; p += KT == 0 ? SK : 1) {
    const FcPart part = parts[blk.first + p];
    switch (part.D) {
      case 1: one(std::integral_constant<int, 1>{}, part); break;
      case 3: one(std::integral_constant<int, 3>{}, part); break;
      default:
        if constexpr (MAXD > 3) one(std::integral_constant<int, 5>{}, part);
    }
  }
  // what this wavefront stores: the four groups of eight columns, or its own one of the shared tile
  constexpr int GROUPS = SK > 1 ? 1 : 4;
  if constexpr (SK > 1) {
    float* fold = reinterpret_cast<float*>(wl);  // 4 KB a wavefront (KT > 0: the region of the weights, which go another way here)
#pragma unroll
    for (int k = 0; k < DR; ++k) {
      __syncthreads();  // (what the region held before is no longer read)
#pragma unroll
      for (int r = 0; r < 16; ++r) fold[(share * 16 + r) * 64 + lane] = acc[k][r];
      __syncthreads();
      if (share < 4)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float sum = fold[(4 * share + e) * 64 + lane];
#pragma unroll
          for (int o = 1; o < SK; ++o) sum += fold[(o * 16 + 4 * share + e) * 64 + lane];
          acc[k][e] = sum;
        }
    }
  }
  if constexpr (DX2 && SK > 1) {  // the row sums of all wavefronts into the first one's (complete: there was a barrier behind the last part)
    float* first = lsum - share * 32 * n2p;
    for (int e = threadIdx.x; e < 32 * n2p; e += 64 * SK) {
      float sum = first[e];
#pragma unroll
      for (int o = 1; o < SK; ++o) sum += first[o * 32 * n2p + e];
      first[e] = sum;
    }
    __syncthreads();
    lsum = first;
    sums = lsum + c * n2p;
  }
  if constexpr (KT == 0) {  // (the straight kernels touch coupled components only)
    float probe = 0.f;
#pragma unroll
    for (int k = 0; k < DR; ++k) {
      if constexpr (SK == 1) probe = fc_probe(acc[k], probe);
      else
#pragma unroll
        for (int e = 0; e < 4; ++e) probe = fmaf(share < 4 ? acc[k][e] : 0.f, 0.f, probe);
    }
    if constexpr (DX2) {
      __builtin_amdgcn_wave_barrier();
      for (int e = h; e < n2; e += 2) probe = fmaf(sums[e], 0.f, probe);
    }
    const bool odd = !(probe == 0.f);
    if (SK > 1 ? __syncthreads_or(odd) : __any(odd)) return false;
  }
  if (z0 + c < Z && share < 4) {
    TI* out = C + z * ldc + blk.c0;
#pragma unroll
    for (int a = 0; a < GROUPS; ++a) {
      const int m = n0 + 8 * (SK > 1 ? share : a) + 4 * h;
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
    for (int e = SK > 1 ? threadIdx.x : lane; e < rows * n2; e += 64 * SK) partial[z0 * n2 + e] = lsum[e / n2 * n2p + e % n2];
  }
  return true;
}

// MAXD: the most components of any block (3 or 5): what the register budget has to hold.
// SK: wavefronts that share a tile.
template <typename TI, int WM, bool MI, bool DX2, int MAXD, int KT, int SK>
__global__ void __launch_bounds__(SK > 4 ? 64 * SK : 256, (MAXD > 3 || KT > 0 || SK > 1 ? 2 : 3)) fc_rows_kernel(const FcBlock* __restrict__ blocks, const FcPart* __restrict__ parts, const float* __restrict__ coef, int nblocks,
                                                         int tiles_n, const TI* __restrict__ A, int64_t lda, const TI* __restrict__ W, const TI* __restrict__ X2,
                                                         int64_t ldx2, const TI* __restrict__ X1, int64_t ldx1, TI* __restrict__ C, int64_t ldc,
                                                         float* __restrict__ partial, int n2, int64_t Z) {
  extern __shared__ __align__(16) float fc_lsum[];  // 16 fragments of weights (KT > 0) or the sums of SK wavefronts, the row sums of every wavefront, its
                                                    // rows of x2 (KT > 0)
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  // four tiles of one row of tiles to a workgroup; with packed weights four rows of tiles under one column: they read the same weights
  // at about the same time
  int64_t zt;
  int column;
  if constexpr (SK > 1) {
    zt = blockIdx.x / tiles_n;
    column = static_cast<int>(blockIdx.x - zt * tiles_n);
  } else if constexpr (WM == kPacked) {
    const int64_t group = blockIdx.x / tiles_n;
    column = static_cast<int>(blockIdx.x - group * tiles_n);
    zt = group * 4 + wave;
  } else {
    const int64_t unit = static_cast<int64_t>(blockIdx.x) * 4 + wave;
    zt = unit / tiles_n;
    column = static_cast<int>(unit - zt * tiles_n);
  }
  int tile = column, b = 0;
  while (b < nblocks && tile >= blocks[b].nt) tile -= blocks[b++].nt;
  const int64_t z0 = zt * 32;
  // (with weights through LDS a wavefront past the last row stays for the barriers: it reads the last row and stores nothing)
  if (b == nblocks || ((KT == 0 || SK > 1) && z0 >= Z)) return;
  const FcBlock blk = blocks[b];
  uint4* wl = reinterpret_cast<uint4*>(fc_lsum);
  float* lsum = fc_lsum + (KT > 0 ? 16 * 64 * 4 : SK > 1 ? SK * 16 * 64 : 0) + wave * 32 * (n2 | 1);
  float* part = DX2 ? partial + static_cast<int64_t>(column) * Z * n2 : nullptr;
  bool whole = true;
  switch (blk.D) {
    case 1: whole = fc_tile<TI, 1, WM, MI, DX2, MAXD, KT, SK>(blk, parts, coef, A, lda, W, X2, ldx2, X1, ldx1, C, ldc, part, lsum, wl, n2, Z, z0, tile * 32); break;
    case 3: whole = fc_tile<TI, 3, WM, MI, DX2, MAXD, KT, SK>(blk, parts, coef, A, lda, W, X2, ldx2, X1, ldx1, C, ldc, part, lsum, wl, n2, Z, z0, tile * 32); break;
    default:
      if constexpr (MAXD > 3) whole = fc_tile<TI, 5, WM, MI, DX2, MAXD, KT, SK>(blk, parts, coef, A, lda, W, X2, ldx2, X1, ldx1, C, ldc, part, lsum, wl, n2, Z, z0, tile * 32);
  }
  if constexpr (KT == 0) {
    if (!whole && (SK == 1 || wave == 0)) fc_tile_coupled<TI>(blocks + b, parts, coef, A, lda, W, X2, ldx2, DX2 ? X1 : nullptr, ldx1, C, ldc, part, lsum, WM, MI, n2, Z, z0, tile * 32);
  }
}

// The weights of every path in the order the matrix instructions take them: fragment (channel of x2, 16 contracted values, 32 columns),
// 16 bytes per lane.
template <typename TI>
__global__ void __launch_bounds__(256) fc_pack_kernel(const FcPack* __restrict__ packs, int npacks, const TI* __restrict__ W, TI* __restrict__ out, int64_t pieces) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= pieces) return;
  int b = 0;
  while (b + 1 < npacks && i >= packs[b].pieces) i -= packs[b++].pieces;
  const FcPack q = packs[b];
  const int nt = (q.N + 31) / 32, lane = static_cast<int>(i & 63), f = static_cast<int>(i >> 6), n = min(f % nt * 32 + (lane & 31), q.N - 1);
  const int kt = f / nt % q.steps, v = f / nt / q.steps;
  const uint16_t* __restrict__ src = reinterpret_cast<const uint16_t*>(W) + q.src + static_cast<int64_t>(v) * q.vs + static_cast<int64_t>(n) * q.sn;
  uint32_t e[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) e[s] = kt * 16 < q.K ? src[static_cast<int64_t>(kt * 16 + (lane >> 5) * 8 + s) * q.sk] : 0;
  *reinterpret_cast<uint4*>(out + q.dst + i * 8) = make_uint4(e[0] | e[1] << 16, e[2] | e[3] << 16, e[4] | e[5] << 16, e[6] | e[7] << 16);
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
  int32_t a0, K, D1, c0, N, D3, coef, j0, d2, nt, ntv;  // nt: 64 x 64 tiles, those of every channel of x2; ntv: across the columns
  int32_t stride, V, js, vs;                            // as in FcPart
  uint32_t mask;
};

// one 64 x 64 tile of the weight gradient of one path and channel of x2, coupled components alone: a column and every other row a lane
template <typename TI>
__device__ __forceinline__ void fc_grad_coupled(const FcGrad* __restrict__ grad, const float* __restrict__ coef, const TI* __restrict__ X1, int64_t ldx1,
                                                          const TI* __restrict__ X2, int64_t ldx2, const TI* __restrict__ G, int64_t ldg, float* __restrict__ P,
                                                          bool mi, int tile, int64_t zb, int64_t ze) {
  const FcGrad q = *grad;
  const int per = q.nt / q.V, channel = tile / per, u0 = tile % per / q.ntv * 64, v0 = tile % per % q.ntv * 64;
  const int c = threadIdx.x & 31, h = (threadIdx.x >> 5) & 1;
#pragma unroll 1
  for (int part = 0; part < 8; ++part) {
    const int v = v0 + 32 * (part & 1) + c, vr = min(v, q.N - 1), ub = u0 + 16 * (part >> 1) + 8 * h;
    float acc[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) acc[r] = 0.f;
#pragma unroll 1
    for (int64_t z = zb; z < ze; ++z) {
      const TI *xr = X1 + z * ldx1 + q.a0, *gr = G + z * ldg + q.c0, *yr = X2 + z * ldx2 + q.j0 + channel * q.vs;
#pragma unroll 1
      for (int i = 0; i < q.D1; ++i) {
        float hv = 0.f;
        for (int k = 0; k < q.D3; ++k) {
          if (!(q.mask >> (i * q.D3 + k) & 1)) continue;
          const float* cf = coef + q.coef + (i * q.D3 + k) * q.d2;
          float s = 0.f;
          for (int j = 0; j < q.d2; ++j) s = fc_coupled(cf[j], fc_widen(yr + j * q.js), s);
          hv = fmaf(s, fc_widen(gr + (mi ? vr * q.D3 + k : k * q.N + vr)), hv);
        }
        if constexpr (sizeof(TI) == 2) hv = mm_widen<TI>(mm_round<TI>(hv));  // (an operand of a product there: of the rows' type)
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const int u = min(ub + r, q.K - 1);
          acc[r] = fmaf(fc_widen(xr + (mi ? u * q.D1 + i : i * q.K + u)), hv, acc[r]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 8; ++r)
      if (v < q.N && ub + r < q.K) P[q.w0 + channel * q.N + static_cast<int64_t>(ub + r) * q.stride + v] = acc[r];
  }
}

template <typename TI, int D1, int D3, bool MI>
__device__ __forceinline__ bool fc_grad_tile(const FcGrad& q, int tile, const float* __restrict__ coef, const TI* __restrict__ X1, int64_t ldx1,
                                             const TI* __restrict__ X2, int64_t ldx2, const TI* __restrict__ G, int64_t ldg, float* __restrict__ P, int64_t zb,
                                             int64_t ze) {
  constexpr int ES = sizeof(TI);
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int per = q.nt / q.V, channel = tile / per;
  tile -= channel * per;
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
    const TI *xr = X1 + zr * ldx1 + q.a0, *gr = G + zr * ldg + q.c0, *yr = X2 + zr * ldx2 + q.j0 + channel * q.vs;
    float s[NI][D3];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int k = 0; k < D3; ++k) s[i][k] = 0.f;
    for (int j = 0; j < q.d2; ++j) {
      const float xj = fc_widen(yr + j * q.js);
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
  float probe = 0.f;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) probe = fc_probe(acc[a][b], probe);
  if (__any(!(probe == 0.f))) return false;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int vv = v0 + 32 * b + c;
      if (vv >= q.N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int uu = u0 + 32 * a + 8 * (r >> 2) + 4 * h + (r & 3);
        if (uu < q.K) P[q.w0 + channel * q.N + static_cast<int64_t>(uu) * q.stride + vv] = acc[a][b][r];
      }
    }
  return true;
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
#define FC_TILE(A, B) whole = fc_grad_tile<TI, A, B, MI>(q, tile, coef, X1, ldx1, X2, ldx2, G, ldg, P, zb, ze)
  bool whole = true;
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
  if (!whole) fc_grad_coupled<TI>(grads + b, coef, X1, ldx1, X2, ldx2, G, ldg, P, MI, tile, zb, ze);
}

// Weight gradient of 2-byte rows where the x2 blocks have several channels: a workgroup takes 64 x 64 of one path for four channels,
// one per wavefront, so that the rows of x1 and of the cotangent - transposed into LDS, 32 at a time, the next ones requested
// meanwhile - serve four channels, and every H_i of a channel serves 64 columns of x1.  54 us for 12 501 rows of 64x0e+64x1o (x)
// 16x0e+16x1o in bfloat16 (73 with the components tested in the loop; 194 with the products of the operands in memory), bound by the
// vector instructions that form H.
constexpr int kDvRows = 32, kDvPad = kDvRows + 8;  // (rows of 80 bytes: 16-byte pieces stay aligned)
template <typename TI, int D1, int D3, int D2, bool MI>
__device__ __forceinline__ void fc_grad_channels(const FcGrad& q, int tile, const float* __restrict__ coef, const TI* __restrict__ X1, int64_t ldx1,
                                                 const TI* __restrict__ X2, int64_t ldx2, const TI* __restrict__ G, int64_t ldg, float* __restrict__ P, int64_t zb,
                                                 int64_t ze, uint16_t* lds) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = lane & 31, h = lane >> 5;
  const int per = q.nt / ((q.V + 3) / 4), v0 = tile / per * 4;  // (nt of this table: 64 x 64 tiles times groups of four channels)
  tile %= per;
  const int u0 = tile / q.ntv * 64, w0 = tile % q.ntv * 64;
  uint16_t *xs = lds, *gs = lds + 3 * 64 * kDvPad;
  float* ys = reinterpret_cast<float*>(lds + 6 * 64 * kDvPad);  // [channel][component][32 rows]
  const FcCoefs cf(coef + q.coef, D1 * D3 * D2);
  fx16 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = fx16{0};

  // staging: this thread's two rows and four columns of every component
  const int pair = tid >> 4, col = 4 * (tid & 15);
  const int uc = min(u0 + col, q.K - 4), wc = min(w0 + col, q.N - 4);
  uint2 rx[2][D1], rg[2][D3];
  float ry[3];  // (4 channels x up to 5 components x 32 rows over 256 threads)
  const int ny = 4 * D2 * kDvRows;
  auto request = [&](int64_t z) {
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int64_t zr = z + 2 * pair + r;
      const bool in = zr < ze;
      const TI *xr = X1 + min(zr, ze - 1) * ldx1 + q.a0, *gr = G + min(zr, ze - 1) * ldg + q.c0;
#pragma unroll
      for (int i = 0; i < D1; ++i) {
        const uint2 t = *reinterpret_cast<const uint2*>(xr + (MI ? uc * D1 + 4 * i : i * q.K + uc));
        rx[r][i] = in ? t : make_uint2(0, 0);
      }
#pragma unroll
      for (int k = 0; k < D3; ++k) {
        const uint2 t = *reinterpret_cast<const uint2*>(gr + (MI ? wc * D3 + 4 * k : k * q.N + wc));
        rg[r][k] = in ? t : make_uint2(0, 0);
      }
    }
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      const int at = tid + 256 * e;
      ry[e] = 0.f;
      if (at < ny) {  // a row's values are adjacent threads' (rows slowest)
        const int row = at / (4 * D2), vj = at - row * (4 * D2), v = vj / D2, j = vj - v * D2;
        if (z + row < ze && v0 + v < q.V) ry[e] = fc_widen(X2 + (z + row) * ldx2 + q.j0 + (v0 + v) * q.vs + j * q.js);
      }
    }
  };
  auto stage = [&](auto dc, uint16_t* to, const auto& regs) {
    constexpr int D = decltype(dc)::value;
    const uint16_t *e0 = reinterpret_cast<const uint16_t*>(&regs[0][0]), *e1 = reinterpret_cast<const uint16_t*>(&regs[1][0]);
#pragma unroll
    for (int m = 0; m < 4 * D; ++m) {
      const int comp = MI ? m % D : m / 4, cc = col + (MI ? m / D : m % 4);
      *reinterpret_cast<uint32_t*>(to + (comp * 64 + cc) * kDvPad + 2 * pair) = static_cast<uint32_t>(e0[m]) | static_cast<uint32_t>(e1[m]) << 16;
    }
  };
  request(zb);
  for (int64_t z = zb; z < ze; z += kDvRows) {
    __syncthreads();
    stage(std::integral_constant<int, D1>{}, xs, rx);
    stage(std::integral_constant<int, D3>{}, gs, rg);
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      const int at = tid + 256 * e;
      if (at < ny) {
        const int row = at / (4 * D2), vj = at - row * (4 * D2);
        ys[vj * kDvRows + row] = ry[e];
      }
    }
    __syncthreads();
    if (z + kDvRows < ze) request(z + kDvRows);
    if (v0 + wave < q.V) {
#pragma unroll 1
      for (int t = 0; t < kDvRows; t += 16) {
        uint4 graw[2][D3];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int k = 0; k < D3; ++k) graw[b][k] = *reinterpret_cast<const uint4*>(gs + (k * 64 + 32 * b + c) * kDvPad + t + 8 * h);
        const float* yv = ys + wave * D2 * kDvRows + t + 8 * h;
#pragma unroll
        for (int i = 0; i < D1; ++i) {
          float H[2][8];
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 8; ++e) H[b][e] = 0.f;
#pragma unroll
          for (int k = 0; k < D3; ++k) {
            if (!fc_couples<D1, D3, D2>(i, k)) continue;
            float s[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) s[e] = 0.f;
#pragma unroll
            for (int j = 0; j < D2; ++j) {
              if (!fc_couples<D1, D3, D2>(i, k, j)) continue;
              const float f = cf[(i * D3 + k) * D2 + j];
              const float4 lo = *reinterpret_cast<const float4*>(yv + j * kDvRows), hi = *reinterpret_cast<const float4*>(yv + j * kDvRows + 4);
              s[0] = fmaf(f, lo.x, s[0]); s[1] = fmaf(f, lo.y, s[1]); s[2] = fmaf(f, lo.z, s[2]); s[3] = fmaf(f, lo.w, s[3]);
              s[4] = fmaf(f, hi.x, s[4]); s[5] = fmaf(f, hi.y, s[5]); s[6] = fmaf(f, hi.z, s[6]); s[7] = fmaf(f, hi.w, s[7]);
            }
#pragma unroll
            for (int b = 0; b < 2; ++b) {
              const uint32_t words[4] = {graw[b][k].x, graw[b][k].y, graw[b][k].z, graw[b][k].w};
#pragma unroll
              for (int e = 0; e < 8; ++e)
                H[b][e] = fmaf(s[e], mm_widen<TI>(static_cast<uint16_t>(e & 1 ? words[e >> 1] >> 16 : words[e >> 1] & 0xffffu)), H[b][e]);
            }
          }
          uint4 hp[2];
#pragma unroll
          for (int b = 0; b < 2; ++b) hp[b] = make_uint4(mm_pack<TI>(H[b][0], H[b][1]), mm_pack<TI>(H[b][2], H[b][3]), mm_pack<TI>(H[b][4], H[b][5]), mm_pack<TI>(H[b][6], H[b][7]));
#pragma unroll
          for (int a = 0; a < 2; ++a) {
            const uint4 xf = *reinterpret_cast<const uint4*>(xs + (i * 64 + 32 * a + c) * kDvPad + t + 8 * h);
#pragma unroll
            for (int b = 0; b < 2; ++b) acc[a][b] = mm_32x32x16<TI>(xf, hp[b], acc[a][b]);
          }
        }
      }
    }
  }
  if (v0 + wave >= q.V) return;
  P += q.w0 + static_cast<int64_t>(v0 + wave) * q.N;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int w = w0 + 32 * b + c;
      if (w >= q.N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int u = u0 + 32 * a + 8 * (r >> 2) + 4 * h + (r & 3);
        if (u < q.K) P[static_cast<int64_t>(u) * q.stride + w] = acc[a][b][r];
      }
    }
}

template <typename TI, bool MI>
__global__ void __launch_bounds__(256, 2) fc_grad_channels_kernel(const FcGrad* __restrict__ grads, const float* __restrict__ coef, int ngrads, int tiles,
                                                                  const TI* __restrict__ X1, int64_t ldx1, const TI* __restrict__ X2, int64_t ldx2,
                                                                  const TI* __restrict__ G, int64_t ldg, float* __restrict__ partial, int64_t numel, int64_t Z,
                                                                  int64_t rows_per_chunk, int64_t chunks) {
  __shared__ __align__(16) uint16_t lds[6 * 64 * kDvPad + 2 * 4 * 5 * kDvRows];
  const int64_t chunk = blockIdx.x / tiles;
  int tile = static_cast<int>(blockIdx.x - chunk * tiles), b = 0;
  if (chunk >= chunks) return;
  while (b < ngrads && tile >= grads[b].nt) tile -= grads[b++].nt;
  if (b == ngrads) return;
  const FcGrad q = grads[b];
  const int64_t zb = chunk * rows_per_chunk, ze = min(zb + rows_per_chunk, Z);
  float* P = partial + chunk * numel;
#define FC_TILE(A, B, C) fc_grad_channels<TI, A, B, C, MI>(q, tile, coef, X1, ldx1, X2, ldx2, G, ldg, P, zb, ze, lds)
  switch (q.D1 * 8 + q.D3) {
    case 9: FC_TILE(1, 1, 1); break;
    case 11: FC_TILE(1, 3, 3); break;
    case 25: FC_TILE(3, 1, 3); break;
    default:
      if (q.d2 == 1) FC_TILE(3, 3, 1);
      else if (q.d2 == 3) FC_TILE(3, 3, 3);
      else FC_TILE(3, 3, 5);
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
    auto factors = [&](auto coupled) {  // of the row, a lane each
      int off = 0;
      __builtin_amdgcn_wave_barrier();
      for (int p = 0; p < ngrads; ++p) {
        const FcGrad q = grads[p];
        const TI* yr = X2 + z * ldx2 + q.j0;
        const int n = q.D1 * q.D3;
        if (lane < n) {
          float f = 0.f;
          for (int j = 0; j < q.d2; ++j) {
            const float cj = coef[q.coef + lane * q.d2 + j], xj = fc_widen(yr + j);
            f = decltype(coupled)::value ? fc_coupled(cj, xj, f) : fmaf(cj, xj, f);
          }
          s[off + lane] = f;
        }
        off += n;
      }
      __builtin_amdgcn_wave_barrier();
    };
    float probe = 0.f;
    auto write = [&](auto coupled) {
      TI* h = H + z * ldh;
      int off = 0;
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
              if (k < q.D3 && (!decltype(coupled)::value || (q.mask >> (i * q.D3 + k) & 1))) {
                const float f = s[off + i * q.D3 + k];
                a = fmaf(f, ga[k], a);
                b = fmaf(f, gb[k], b);
              }
            probe = fmaf(a, 0.f, fmaf(b, 0.f, probe));
            store2(h + i * q.N + w, a, b);
          }
        }
        h += q.D1 * q.N;
        off += q.D1 * q.D3;
      }
    };
    factors(std::false_type{});
    write(std::false_type{});
    if (__any(!(probe == 0.f))) {  // (not finite: again, coupled components alone)
      factors(std::true_type{});
      write(std::true_type{});
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

static_assert(sizeof(FcPart) == 56 && sizeof(FcBlock) == 24 && sizeof(FcGrad) == 72 && sizeof(FcPack) == 48, "the tables the host uploads");

#define FC_DISPATCH(dt, CALL)                                      \
  do {                                                             \
    if ((dt) == CUEQ_F32) { CALL(float); }                         \
    else if ((dt) == CUEQ_F16) { CALL(f16bits); }                  \
    else { CALL(uint16_t); }                                       \
  } while (0)

// gradient == 0: rows of x1 against W; 1: rows of the cotangent against W^T, and with X1, partial and dX2 given also the gradient of x2
// packed > 0: W holds the packed weights (2-byte elements) in groups of 2 or 4 steps of 16 contracted values (blocks held in registers, the
// couplings of fc_couples only), or - 5 - in as many as every block has
extern "C" int cueq_fc_flex(int32_t dtype, int32_t gradient, int32_t mul_ir, int32_t packed, int64_t rows, const void* A, int64_t lda, const void* W, const void* X2, int64_t ldx2,
                            const void* X1, int64_t ldx1, void* C, int64_t ldc, const void* blocks, int32_t nblocks, const void* parts, const float* coef,
                            int32_t column_tiles, int32_t most_components, int32_t n2, float* partial, void* dX2, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  CUEQ_REQUIRE(dtype == CUEQ_F32 || dtype == CUEQ_BF16 || dtype == CUEQ_F16, CUEQ_ERR_UNSUPPORTED, "fc_flex: dtype must be float32, bfloat16 or half");
  CUEQ_REQUIRE(rows >= 0 && nblocks > 0 && column_tiles > 0 && n2 > 0 && n2 <= 128, CUEQ_ERR_INVALID, "fc_flex: bad extents");
  CUEQ_REQUIRE(!packed || dtype != CUEQ_F32, CUEQ_ERR_UNSUPPORTED, "fc_flex: packed weights are 2-byte elements");
  if (rows == 0) return CUEQ_OK;
  CUEQ_REQUIRE(A && W && X2 && C && blocks && parts && coef && (!dX2 || (gradient && X1 && partial)), CUEQ_ERR_INVALID, "fc_flex: null operand");
  const int64_t epv = dtype == CUEQ_F32 ? 4 : 8;
  CUEQ_REQUIRE(((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(C) | reinterpret_cast<uintptr_t>(W) | reinterpret_cast<uintptr_t>(X1)) & 15) == 0 &&
                   lda % epv == 0 && ldc % epv == 0 && ldx1 % epv == 0,
               CUEQ_ERR_UNSUPPORTED, "fc_flex: rows must be 16-byte aligned");
  const int64_t row_tiles = (rows + 31) / 32;
  const bool held = packed && packed <= 4 && most_components <= 3;  // (source blocks in registers, channel by channel)
  // Few tiles: eight (four) wavefronts share one, each with some of its parts (held: of the channels).  A tile is one serial chain over the
  // paths and channels, 150 us for float and 16 channels, and four times fewer rows took no less.  Shared, a CU takes one tile at a time:
  // how many rounds of that a chain is worth goes with its parts, and one part cannot be shared.  us for one / shared, 64 channels, forward +
  // input gradients unless said otherwise, by parts of a block and tiles a CU:
  //   0e+1o blocks, float: (x) 0e, 1 part, forward 1 10.7 / 12.2; 0e+1o, 2, forward 1 13.5 / 12.1, 2 14.4 / 20.6; l <= 2, 2.5, forward 1
  //   19.9 / 13.4, 1.5 19.7 / 22.1; 2 channels, 4, 2 55 / 50, 3 57 / 69; 4 channels, 8, 3 103 / 84, 4 102 / 109; 8 channels, 16, 6 275 / 246, 8
  //   293 / 321 (32 (x) 8 6 180 / 179); 16 channels, 32, 6 540 / 435, 8 575 / 575
  //   0e+1o+2e blocks (a SIMD holds fewer tiles): (x) 0e, 1, 0.75 36 / 38; 0e+1o, 2.3, 0.75 56 / 41, 1.5 57 / 71; l <= 2, 3.7, 1.5 93 / 81, 3 103 / 123,
  //   bfloat16 66 / 62, 3 68 / 94; l <= 3, 4.3, 2.2 118 / 112, 3 124 / 138; 2 channels l <= 2, 7.3, 3 186 / 150, 12 472 / 462, 18 651 / 674; 4
  //   channels, 15, 12 925 / 719, bfloat16 575 / 487
  //   held: 2 channels 2 37 / 35, 3 42 / 56; 16 channels 4 138 / 136; 4 channels 2 43 / 43, 3 47 / 70
  const int64_t tiles = row_tiles * column_tiles;
  const int said = mul_ir >> 1;
  mul_ir &= 1;
  const int rounds = held ? 2 : said == 0 ? 3 : said < 2 ? 0 : most_components > 3 ? (said < 3 ? 1 : said < 6 ? 2 : 12) : said < 4 ? 1 : said < 8 ? 2 : said < 16 ? 3 : 6;
  const int share = tiles > static_cast<int64_t>(rounds) * device_cus() ? 1 : held ? 4 : n2 <= 64 ? 8 : 1;  // (n2: 100 KB of LDS)
  const int64_t grid = share > 1 ? row_tiles * column_tiles : packed ? (row_tiles + 3) / 4 * column_tiles : (row_tiles * column_tiles + 3) / 4;
  CUEQ_REQUIRE(grid < (1ll << 31), CUEQ_ERR_TOO_LARGE, "fc_flex: too many rows");
  const size_t lds = (dX2 ? std::max(4, share) * 32 * (n2 | 1) * sizeof(float) : 0) +
                     (held ? 16 * 1024 + 4 * 32 * fc_x2_words(n2) * sizeof(uint32_t) : share > 1 ? share * 16 * 64 * sizeof(float) : 0);
  // (the timing label says whether tiles are shared, so a test can tell which kernel a shape ran on)
  KernelTimer timer(gradient ? (share > 1 ? "fc_flex_dx_shared" : "fc_flex_dx") : share > 1 ? "fc_flex_fwd_shared" : "fc_flex_fwd", stream);
#define FC_GD(TI, WM, MI, DX, MD, KT)                                                                                                            \
  do {                                                                                                                                         \
    if (share > 1) FC_GE(TI, WM, MI, DX, MD, KT, (KT > 0 ? 4 : 8));                                                                            \
    else FC_GE(TI, WM, MI, DX, MD, KT, 1);                                                                                                     \
  } while (0)
#define FC_GE(TI, WM, MI, DX, MD, KT, SK)                                                                                                            \
  do {                                                                                                                                         \
    if (lds > 64 * 1024)                                                                                                                       \
      CUEQ_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(fc_rows_kernel<TI, WM, MI, DX, MD, KT, SK>),                                \
                                         hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));                                  \
    FC_GL(TI, WM, MI, DX, MD, KT, SK);                                                                                                             \
  } while (0)
#define FC_GL(TI, WM, MI, DX, MD, KT, SK) hipLaunchKernelGGL((fc_rows_kernel<TI, WM, MI, DX, MD, KT, SK>), dim3(static_cast<unsigned>(grid)), dim3(SK > 4 ? 64 * SK : 256), lds, stream, static_cast<const FcBlock*>(blocks), static_cast<const FcPart*>(parts), coef, nblocks, column_tiles, static_cast<const TI*>(A), lda, static_cast<const TI*>(W), static_cast<const TI*>(X2), ldx2, static_cast<const TI*>(X1), ldx1, static_cast<TI*>(C), ldc, partial, n2, rows)
#define FC_GK(TI, MI, DX)                                              \
  do {                                                                 \
    if constexpr (sizeof(TI) == 2) {                                   \
      if (most_components > 3) FC_GD(TI, kPacked, MI, DX, 5, 0);       \
      else if (packed > 4) FC_GD(TI, kPacked, MI, DX, 3, 0);           \
      else if (packed > 2) FC_GD(TI, kPacked, MI, DX, 3, 4);           \
      else FC_GD(TI, kPacked, MI, DX, 3, 2);                           \
    }                                                                  \
  } while (0)
#define FC_GO(TI, WM, MI, DX)                                          \
  do {                                                                 \
    if (packed) FC_GK(TI, MI, DX);                                     \
    else if (most_components <= 3) FC_GD(TI, WM, MI, DX, 3, 0);        \
    else FC_GD(TI, WM, MI, DX, 5, 0);                                  \
  } while (0)
#define FC(TI)                                                                                                    \
  do {                                                                                                            \
    if (!gradient) { if (mul_ir) FC_GO(TI, kPlain, true, false); else FC_GO(TI, kPlain, false, false); }          \
    else if (dX2) { if (mul_ir) FC_GO(TI, kTransposed, true, true); else FC_GO(TI, kTransposed, false, true); }   \
    else { if (mul_ir) FC_GO(TI, kTransposed, true, false); else FC_GO(TI, kTransposed, false, false); }          \
  } while (0)
  FC_DISPATCH(dtype, FC);
#undef FC
#undef FC_GO
#undef FC_GK
#undef FC_GD
#undef FC_GE
#undef FC_GL
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

// the weights as cueq_fc_flex takes them with `packed`: pieces of 16 bytes, those of all paths of the table
extern "C" int cueq_fc_pack(int32_t dtype, const void* W, void* out, const void* packs, int32_t npacks, int64_t pieces, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  CUEQ_REQUIRE(dtype == CUEQ_BF16 || dtype == CUEQ_F16, CUEQ_ERR_UNSUPPORTED, "fc_pack: dtype must be bfloat16 or half");
  CUEQ_REQUIRE(npacks > 0 && pieces > 0 && pieces < (1ll << 31) && W && out && packs, CUEQ_ERR_INVALID, "fc_pack: bad extents or null operand");
  KernelTimer timer("fc_pack", stream);
  hipLaunchKernelGGL(fc_pack_kernel<uint16_t>, dim3(static_cast<unsigned>((pieces + 255) / 256)), dim3(256), 0, stream, static_cast<const FcPack*>(packs), npacks,
                     static_cast<const uint16_t*>(W), static_cast<uint16_t*>(out), pieces);
  CUEQ_CHECK_HIP(hipGetLastError());
  return CUEQ_OK;
}

// partial products of every path's weight gradient: cueq_fc_flex_dw_chunks x numel floats, to be summed in order (cueq_sum_runs)
// (by_channels: fc_grad_channels_kernel, a workgroup per tile and chunk - two for every CU -, else a wavefront)
static int64_t fc_rows_per_chunk(int64_t rows, int32_t tiles, bool by_channels) {
  const int64_t step = by_channels ? kDvRows : 16;
  int64_t chunks = std::min<int64_t>((by_channels ? 2ll : 8ll) * device_cus() / std::max(1, tiles), (rows + step - 1) / step);
  chunks = std::max<int64_t>(1, chunks);
  return ((rows + chunks - 1) / chunks + step - 1) / step * step;
}
extern "C" int64_t cueq_fc_flex_dw_chunks(int64_t rows, int32_t tiles, int32_t by_channels) {
  const int64_t rpc = fc_rows_per_chunk(rows, tiles, by_channels != 0);
  return (rows + rpc - 1) / rpc;
}
extern "C" int cueq_fc_flex_dw(int32_t dtype, int32_t mul_ir, int32_t by_channels, int64_t rows, const void* X1, int64_t ldx1, const void* X2, int64_t ldx2,
                               const void* G, int64_t ldg, const void* grads, int32_t ngrads, const float* coef, int32_t tiles, int64_t numel, float* partial,
                               void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  CUEQ_REQUIRE(dtype == CUEQ_F32 || dtype == CUEQ_BF16 || dtype == CUEQ_F16, CUEQ_ERR_UNSUPPORTED, "fc_flex_dw: dtype must be float32, bfloat16 or half");
  CUEQ_REQUIRE(rows > 0 && ngrads > 0 && tiles > 0 && numel > 0, CUEQ_ERR_INVALID, "fc_flex_dw: bad extents");
  CUEQ_REQUIRE(X1 && X2 && G && grads && coef && partial, CUEQ_ERR_INVALID, "fc_flex_dw: null operand");
  CUEQ_REQUIRE(!by_channels || (dtype != CUEQ_F32 && ((reinterpret_cast<uintptr_t>(X1) | reinterpret_cast<uintptr_t>(G)) & 7) == 0 && ldx1 % 4 == 0 && ldg % 4 == 0),
               CUEQ_ERR_UNSUPPORTED, "fc_flex_dw: channels together need 2-byte rows in 8-byte pieces");
  const int64_t rpc = fc_rows_per_chunk(rows, tiles, by_channels != 0), chunks = (rows + rpc - 1) / rpc;
  const int64_t grid = by_channels ? chunks * tiles : (chunks * tiles + 3) / 4;
  CUEQ_REQUIRE(grid < (1ll << 31), CUEQ_ERR_TOO_LARGE, "fc_flex_dw: too many tiles");
  KernelTimer timer("fc_flex_dw", stream);
#define FC_GO(KERNEL, TI, MI) hipLaunchKernelGGL((KERNEL<TI, MI>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, static_cast<const FcGrad*>(grads), coef, ngrads, tiles, static_cast<const TI*>(X1), ldx1, static_cast<const TI*>(X2), ldx2, static_cast<const TI*>(G), ldg, partial, numel, rows, rpc, chunks)
#define FC_CHANNELS(TI) do { if (mul_ir) FC_GO(fc_grad_channels_kernel, TI, true); else FC_GO(fc_grad_channels_kernel, TI, false); } while (0)
#define FC(TI) do { if (mul_ir) FC_GO(fc_grad_kernel, TI, true); else FC_GO(fc_grad_kernel, TI, false); } while (0)
  if (by_channels) {
    if (dtype == CUEQ_F16) FC_CHANNELS(f16bits);
    else FC_CHANNELS(uint16_t);
  } else {
    FC_DISPATCH(dtype, FC);
  }
#undef FC
#undef FC_CHANNELS
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
