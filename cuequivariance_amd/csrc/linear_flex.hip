// Equivariant Linear (uv,iu,iv) for batches that do not fill the chip with the row-streaming kernels (linear_rows*.hip: all
// weights of a launch in LDS, one block per CU, one wavefront per 32 rows and whole column block), and for shapes those do not
// take: any number of input blocks per output block, extents that are multiples of 8 (float) or 16 (2-byte), rows in ir_mul or
// mul_ir.  One launch computes every block of the result, one the partial products of every weight block.
//
//   out[z, c0 + v D + i] = sum over the parts p of the block  coeff_p sum_u A[z, a_p + u D + i] W_p[u, v]
//
// What bounds them: at a few thousand rows the latency of one wavefront's serial chain, so the unit of work is a tile of 32 rows
// and 32 columns (the row-streaming kernels give a wavefront 32 x 128), without LDS and without barriers.  The products are
// issued as W-columns x rows: a lane then holds one row and, per accumulator, 4 adjacent columns of it (times D components in
// mul_ir), and both its loads and its stores are whole 16-byte pieces; the k order inside a step is free, so a lane takes 4 (8)
// adjacent channels of its row.  (Forward of 5 003 rows of 128x0e+128x1o+128x2e in mul_ir, float: 131 us in three row-streaming
// launches, 40 us here.)  The wavefronts of a block share the rows and differ in the columns: the rows come from L1 for
// all but the first.
#include <algorithm>

#include "common.h"
#include "cw_common.h"
#include "u1d_spec.h"

namespace cueq {
namespace {

struct FlexPart {   // one K x N weight block applied to one input block
  int64_t a0, w0;
  int32_t K;
  float coeff;
};
struct FlexBlock {  // one block of the result
  int64_t c0;
  int32_t N, D, first, parts, nt, unused;  // nt: column tiles
};

typedef float fx16 __attribute__((ext_vector_type(16)));

// one tile: rows z0 .. z0 + 32 ZT, columns n0 .. n0 + 32 of the block.  WT: the weights are read transposed (input gradient).
// SK: wavefronts that share the tile, each with its part of every contraction; the first adds the others' sums, in order, through
// LDS and stores (SK > 1: all SK wavefronts of the workgroup are here).
template <typename TI, int D, int ZT, bool WT, int SK>
__device__ __forceinline__ void flex_tile(const FlexBlock& blk, const FlexPart* __restrict__ parts, const TI* __restrict__ A, int64_t lda, const TI* __restrict__ W,
                                          TI* __restrict__ C, int64_t ldc, int64_t Z, int64_t z0, int n0) {
  constexpr int ES = sizeof(TI), EPV = 16 / ES, STEP = 2 * EPV;  // channels per step: 4 + 4 (float), 8 + 8
  static_assert(SK == 1 || ZT == 1, "a shared tile has 32 rows");
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int share = SK > 1 ? __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)) : 0;
  fx16 acc[ZT][D];
#pragma unroll
  for (int t = 0; t < ZT; ++t)
#pragma unroll
    for (int i = 0; i < D; ++i) acc[t][i] = fx16{0};
  const int n = min(n0 + c, blk.N - 1);
  const TI* row[ZT];
#pragma unroll
  for (int t = 0; t < ZT; ++t) row[t] = A + min(z0 + 32 * t + c, Z - 1) * lda;
  float scale = 1.0f;
  for (int p = 0; p < blk.parts; ++p) {
    const FlexPart part = parts[blk.first + p];
    if (p && part.coeff != scale) {  // (what is summed so far counts in units of the coefficient)
      const float f = scale / part.coeff;
#pragma unroll
      for (int t = 0; t < ZT; ++t)
#pragma unroll
        for (int i = 0; i < D; ++i) acc[t][i] *= f;
    }
    scale = part.coeff;
    uint4 x[ZT][D], xn[ZT][D];
    uint4 wv, wn;
    auto load = [&](int k0, uint4 (&xx)[ZT][D], uint4& ww) {
      const int k = k0 + EPV * h;
#pragma unroll
      for (int t = 0; t < ZT; ++t)
#pragma unroll
        for (int i = 0; i < D; ++i) xx[t][i] = *reinterpret_cast<const uint4*>(row[t] + part.a0 + static_cast<int64_t>(k) * D + i * EPV);
      if constexpr (WT) {
        ww = *reinterpret_cast<const uint4*>(W + part.w0 + static_cast<int64_t>(n) * part.K + k);
      } else if constexpr (ES == 4) {
        uint32_t e[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) e[s] = reinterpret_cast<const uint32_t*>(W)[part.w0 + static_cast<int64_t>(k + s) * blk.N + n];
        ww = make_uint4(e[0], e[1], e[2], e[3]);
      } else {
        uint32_t e[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) e[s] = reinterpret_cast<const uint16_t*>(W)[part.w0 + static_cast<int64_t>(k + s) * blk.N + n];
        ww = make_uint4(e[0] | e[1] << 16, e[2] | e[3] << 16, e[4] | e[5] << 16, e[6] | e[7] << 16);
      }
    };
    const int steps = part.K / STEP, first = SK > 1 ? steps * share / SK * STEP : 0, last = SK > 1 ? steps * (share + 1) / SK * STEP : part.K;
    if (SK > 1 && first == last) continue;
    load(first, x, wv);
    for (int k0 = first; k0 < last; k0 += STEP) {
      load(min(k0 + STEP, last - STEP), xn, wn);
#pragma unroll
      for (int t = 0; t < ZT; ++t) {
        if constexpr (ES == 4) {
          const float* xf = reinterpret_cast<const float*>(&x[t][0]);
          const float* wf = reinterpret_cast<const float*>(&wv);
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < D; ++i) acc[t][i] = __builtin_amdgcn_mfma_f32_32x32x2f32(wf[s], xf[s * D + i], acc[t][i], 0, 0, 0);
        } else {
#pragma unroll
          for (int i = 0; i < D; ++i) {
            uint4 op;
            if constexpr (D == 1) op = x[t][0];
            else op = make_uint4(mm_pick(&x[t][0], i, D + i), mm_pick(&x[t][0], 2 * D + i, 3 * D + i), mm_pick(&x[t][0], 4 * D + i, 5 * D + i),
                                 mm_pick(&x[t][0], 6 * D + i, 7 * D + i));
            acc[t][i] = mm_32x32x16<TI>(wv, op, acc[t][i]);
          }
        }
      }
#pragma unroll
      for (int t = 0; t < ZT; ++t)
#pragma unroll
        for (int i = 0; i < D; ++i) x[t][i] = xn[t][i];
      wv = wn;
    }
  }
  if constexpr (SK > 1) {
    __shared__ float others[SK - 1][16][64];
#pragma unroll
    for (int i = 0; i < D; ++i) {
      if (share)
#pragma unroll
        for (int r = 0; r < 16; ++r) others[share - 1][r][lane] = acc[0][i][r];
      __syncthreads();
      if (!share)
#pragma unroll
        for (int r = 0; r < 16; ++r)
#pragma unroll
          for (int o = 0; o < SK - 1; ++o) acc[0][i][r] += others[o][r][lane];
      __syncthreads();
    }
    if (share) return;
  }
#pragma unroll
  for (int t = 0; t < ZT; ++t) {
    const int64_t z = z0 + 32 * t + c;
    if (z >= Z) continue;
    TI* out = C + z * ldc + blk.c0;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int m = n0 + 8 * a + 4 * h;  // four adjacent columns, D components each
      if (m >= blk.N) continue;
      float v[4 * D];
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < D; ++i) v[b * D + i] = scale * acc[t][i][4 * a + b];
      if constexpr (ES == 4) {
#pragma unroll
        for (int i = 0; i < D; ++i) *reinterpret_cast<float4*>(out + m * D + 4 * i) = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
      } else {
#pragma unroll
        for (int i = 0; i < D; ++i)
          *reinterpret_cast<uint2*>(out + m * D + 4 * i) = make_uint2(mm_pack<TI>(v[4 * i], v[4 * i + 1]), mm_pack<TI>(v[4 * i + 2], v[4 * i + 3]));
      }
    }
  }
}

// unit = (column tiles of the blocks one after the other) x (row tile); the column tile runs fastest, so a block's wavefronts share rows
// (SK > 1: a workgroup per unit)
template <typename TI, bool WT, int ZBIG, int SK>
__global__ void __launch_bounds__(256, 2) flex_rows_kernel(const FlexBlock* __restrict__ blocks, const FlexPart* __restrict__ parts, int nblocks, int tiles_n,
                                                           const TI* __restrict__ A, int64_t lda, const TI* __restrict__ W, TI* __restrict__ C, int64_t ldc,
                                                           int64_t Z) {
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int64_t unit = SK > 1 ? static_cast<int64_t>(blockIdx.x) : static_cast<int64_t>(blockIdx.x) * 4 + wave;
  const int64_t zt = unit / tiles_n;
  int tile = static_cast<int>(unit - zt * tiles_n);
  int b = 0;
  while (b < nblocks && tile >= blocks[b].nt) tile -= blocks[b++].nt;
  constexpr int RZ = 32 * ZBIG;
  const int64_t z0 = zt * RZ;
  if (b == nblocks || z0 >= Z) return;
  const FlexBlock blk = blocks[b];
  switch (blk.D) {
    case 1: flex_tile<TI, 1, ZBIG, WT, SK>(blk, parts, A, lda, W, C, ldc, Z, z0, tile * 32); break;
    case 3:
      for (int t = 0; t < ZBIG && z0 + 32 * t < Z; ++t) flex_tile<TI, 3, 1, WT, SK>(blk, parts, A, lda, W, C, ldc, Z, z0 + 32 * t, tile * 32);
      break;
    case 5:
      for (int t = 0; t < ZBIG && z0 + 32 * t < Z; ++t) flex_tile<TI, 5, 1, WT, SK>(blk, parts, A, lda, W, C, ldc, Z, z0 + 32 * t, tile * 32);
      break;
    default:
      for (int t = 0; t < ZBIG && z0 + 32 * t < Z; ++t) flex_tile<TI, 7, 1, WT, SK>(blk, parts, A, lda, W, C, ldc, Z, z0 + 32 * t, tile * 32);
  }
}

// Weight gradients: dW[w0 + u N + v] = coeff sum_z sum_i x[z, a0 + i sa + u D + i'] g[z, c0 + i sc + v D + i'] over a chunk of rows,
// a wavefront per (block, 64 x 64 tile, chunk); partial[chunk][weight], summed in order afterwards.
struct FlexGrad {
  int64_t a0, c0, w0;
  int32_t K, N, D, comps, sa, sc, nt, ntv;  // D > 1: components interleaved (mul_ir), else `comps` components at strides sa, sc
  float coeff;
};

// NT x NT tiles of 32 x 32: one for blocks of at most 32 channels (a 64 x 64 tile would be three quarters padding), four otherwise
template <typename TI, int D, int NT>
__device__ __forceinline__ void flex_grad_tile(const FlexGrad& q, int tile, const TI* __restrict__ X, int64_t ldx, const TI* __restrict__ G, int64_t ldg,
                                               float* __restrict__ P, int64_t zb, int64_t ze) {
  constexpr int ES = sizeof(TI), ROWS = ES == 4 ? 2 : 16;  // rows (contraction) per matrix instruction
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int u0 = (tile / q.ntv) * 64, v0 = (tile % q.ntv) * 64;
  fx16 acc[NT][NT];
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = fx16{0};
  int u[NT], v[NT];
#pragma unroll
  for (int a = 0; a < NT; ++a) {
    u[a] = min(u0 + 32 * a + c, q.K - 1);
    v[a] = min(v0 + 32 * a + c, q.N - 1);
  }
  for (int comp = 0; comp < q.comps; ++comp) {
    const TI *xp = X + q.a0 + static_cast<int64_t>(comp) * q.sa, *gp = G + q.c0 + static_cast<int64_t>(comp) * q.sc;
    if constexpr (ES == 4) {
      constexpr int U = D == 1 ? 8 : D == 3 ? 4 : 2;  // row pairs in flight
      for (int64_t z = zb; z < ze; z += 2 * U) {
        float xa[U][NT][D], ga[U][NT][D];
#pragma unroll
        for (int s = 0; s < U; ++s) {
          const int64_t zz = z + 2 * s + h, zr = min(zz, ze - 1);
#pragma unroll
          for (int a = 0; a < NT; ++a)
#pragma unroll
            for (int i = 0; i < D; ++i) {
              const float xv = xp[zr * ldx + u[a] * D + i], gv = gp[zr * ldg + v[a] * D + i];
              xa[s][a][i] = zz < ze ? xv : 0.f;  // (rows past the chunk count nothing)
              ga[s][a][i] = zz < ze ? gv : 0.f;
            }
        }
#pragma unroll
        for (int s = 0; s < U; ++s)
#pragma unroll
          for (int i = 0; i < D; ++i)
#pragma unroll
            for (int a = 0; a < NT; ++a)
#pragma unroll
              for (int b = 0; b < NT; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(xa[s][a][i], ga[s][b][i], acc[a][b], 0, 0, 0);
      }
    } else {
      const uint16_t *xq = reinterpret_cast<const uint16_t*>(xp), *gq = reinterpret_cast<const uint16_t*>(gp);
      for (int64_t z = zb; z < ze; z += ROWS) {
#pragma unroll 1
        for (int i = 0; i < D; ++i) {
          uint4 xa[NT], ga[NT];
#pragma unroll
          for (int a = 0; a < NT; ++a) {
            uint32_t ex[8], eg[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) {
              const int64_t zz = z + 8 * h + s, zr = min(zz, ze - 1);
              const uint32_t xv = xq[zr * ldx + u[a] * D + i], gv = gq[zr * ldg + v[a] * D + i];
              ex[s] = zz < ze ? xv : 0u;
              eg[s] = zz < ze ? gv : 0u;
            }
            xa[a] = make_uint4(ex[0] | ex[1] << 16, ex[2] | ex[3] << 16, ex[4] | ex[5] << 16, ex[6] | ex[7] << 16);
            ga[a] = make_uint4(eg[0] | eg[1] << 16, eg[2] | eg[3] << 16, eg[4] | eg[5] << 16, eg[6] | eg[7] << 16);
          }
#pragma unroll
          for (int a = 0; a < NT; ++a)
#pragma unroll
            for (int b = 0; b < NT; ++b) acc[a][b] = mm_32x32x16<TI>(xa[a], ga[b], acc[a][b]);
        }
      }
    }
  }
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) {
      const int vv = v0 + 32 * b + c;
      if (vv >= q.N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int uu = u0 + 32 * a + 8 * (r >> 2) + 4 * h + (r & 3);
        if (uu < q.K) P[q.w0 + static_cast<int64_t>(uu) * q.N + vv] = q.coeff * acc[a][b][r];
      }
    }
}

template <typename TI>
__global__ void __launch_bounds__(256, 2) flex_grad_kernel(const FlexGrad* __restrict__ grads, int ngrads, int tiles, const TI* __restrict__ X, int64_t ldx,
                                                           const TI* __restrict__ G, int64_t ldg, float* __restrict__ partial, int64_t numel, int64_t Z,
                                                           int64_t rows_per_chunk, int64_t chunks) {
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int64_t unit = static_cast<int64_t>(blockIdx.x) * 4 + wave;
  const int64_t chunk = unit / tiles;
  if (chunk >= chunks) return;
  int tile = static_cast<int>(unit - chunk * tiles), b = 0;
  while (b < ngrads && tile >= grads[b].nt) tile -= grads[b++].nt;
  if (b == ngrads) return;
  const FlexGrad q = grads[b];
  const int64_t zb = chunk * rows_per_chunk, ze = min(zb + rows_per_chunk, Z);
  float* P = partial + chunk * numel;
#define FLEX_TILE(D) do { if (q.K <= 32 && q.N <= 32) flex_grad_tile<TI, D, 1>(q, tile, X, ldx, G, ldg, P, zb, ze); else flex_grad_tile<TI, D, 2>(q, tile, X, ldx, G, ldg, P, zb, ze); } while (0)
  switch (q.D) {
    case 1: FLEX_TILE(1); break;
    case 3: FLEX_TILE(3); break;
    case 5: FLEX_TILE(5); break;
    default: FLEX_TILE(7);
  }
#undef FLEX_TILE
}

// out[w] = sum over the chunks, in order, rounded once to the weights' type; 16 chunk lanes x 64 weights per block
template <typename TO>
__global__ void __launch_bounds__(1024) flex_sum_kernel(const float* __restrict__ in, TO* __restrict__ out, int64_t chunks, int64_t numel) {
  __shared__ float part[16][64];
  const int cl = threadIdx.x & 63, rl = threadIdx.x >> 6;
  const int64_t w = static_cast<int64_t>(blockIdx.x) * 64 + cl;
  float s = 0;
  if (w < numel) {
    int64_t r = rl;
    for (; r + 48 < chunks; r += 64) {
      const float v0 = in[r * numel + w], v1 = in[(r + 16) * numel + w], v2 = in[(r + 32) * numel + w], v3 = in[(r + 48) * numel + w];
      s += v0; s += v1; s += v2; s += v3;
    }
    for (; r < chunks; r += 16) s += in[r * numel + w];
  }
  part[rl][cl] = s;
  __syncthreads();
  if (rl == 0 && w < numel) {
    float total = 0;
#pragma unroll
    for (int t = 0; t < 16; ++t) total += part[t][cl];
    if constexpr (sizeof(TO) == 4) out[w] = total;
    else reinterpret_cast<uint16_t*>(out)[w] = mm_round<TO>(total);
  }
}

// The same sum where a weight block has rows of its own: block b of `per` weights = rows first[b] .. first[b + 1] of in.
struct RunTable {
  int32_t first[33];
  int64_t w0[32];
};
template <typename TO>
__global__ void __launch_bounds__(1024) run_sum_kernel(const float* __restrict__ in, TO* __restrict__ out, RunTable runs, int per) {
  __shared__ float part[16][64];
  const int cl = threadIdx.x & 63, rl = threadIdx.x >> 6, b = blockIdx.y;
  const int w = static_cast<int>(blockIdx.x) * 64 + cl, end = runs.first[b + 1];
  float s = 0;
  if (w < per) {
    int r = runs.first[b] + rl;
    const float* p = in + w;
    for (; r + 48 < end; r += 64) {
      const float v0 = p[static_cast<int64_t>(r) * per], v1 = p[static_cast<int64_t>(r + 16) * per], v2 = p[static_cast<int64_t>(r + 32) * per],
                  v3 = p[static_cast<int64_t>(r + 48) * per];
      s += v0; s += v1; s += v2; s += v3;
    }
    for (; r < end; r += 16) s += p[static_cast<int64_t>(r) * per];
  }
  part[rl][cl] = s;
  __syncthreads();
  if (rl == 0 && w < per) {
    float total = 0;
#pragma unroll
    for (int t = 0; t < 16; ++t) total += part[t][cl];
    if constexpr (sizeof(TO) == 4) out[runs.w0[b] + w] = total;
    else reinterpret_cast<uint16_t*>(out)[runs.w0[b] + w] = mm_round<TO>(total);
  }
}

}  // namespace
}  // namespace cueq

using namespace cueq;

static_assert(sizeof(FlexPart) == 24 && sizeof(FlexBlock) == 32 && sizeof(FlexGrad) == 64, "the tables the host uploads");

#define FLEX_DISPATCH(dt, CALL)                                    \
  do {                                                             \
    if ((dt) == CUEQ_F32) { CALL(float); }                         \
    else if ((dt) == CUEQ_F16) { CALL(f16bits); }                  \
    else { CALL(uint16_t); }                                       \
  } while (0)

extern "C" int cueq_linear_flex(int32_t dtype, int32_t transposed_weights, int64_t rows, const void* A, int64_t lda, const void* W, void* C, int64_t ldc,
                                const void* blocks, int32_t nblocks, const void* parts, int32_t column_tiles, int32_t mul_ir, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  CUEQ_REQUIRE(dtype == CUEQ_F32 || dtype == CUEQ_BF16 || dtype == CUEQ_F16, CUEQ_ERR_UNSUPPORTED, "linear_flex: dtype must be float32, bfloat16 or half");
  CUEQ_REQUIRE(rows >= 0 && nblocks > 0 && column_tiles > 0, CUEQ_ERR_INVALID, "linear_flex: bad extents");
  if (rows == 0) return CUEQ_OK;
  CUEQ_REQUIRE(A && W && C && blocks && parts, CUEQ_ERR_INVALID, "linear_flex: null operand");
  const int64_t es = dtype == CUEQ_F32 ? 4 : 2, epv = 16 / es;
  CUEQ_REQUIRE(((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(C) | reinterpret_cast<uintptr_t>(W)) & 15) == 0 && lda % epv == 0 && ldc % epv == 0,
               CUEQ_ERR_UNSUPPORTED, "linear_flex: rows must be 16-byte aligned");
  // two row tiles per wavefront halve the weight loads once there are units enough for two per SIMD
  const int64_t zt1 = (rows + 31) / 32;
  const bool big = zt1 * column_tiles >= 8 * 4ll * device_cus();
  // four wavefronts share a tile where all tiles, four wavefronts each, still run at once (two workgroups to a CU): 300 rows of
  // 128x0e+128x1o+128x2e in mul_ir, float, forward 21.8 -> 9.7 us, 1 000 rows 22.1 -> 12.6 (1 400 rows, past the line: 22.5 either way)
  const bool shared = zt1 * column_tiles <= 2ll * device_cus();
  const int64_t units = (big ? (rows + 63) / 64 : zt1) * column_tiles, grid = shared ? units : (units + 3) / 4;
  CUEQ_REQUIRE(grid < (1ll << 31), CUEQ_ERR_TOO_LARGE, "linear_flex: too many rows");
  KernelTimer timer(mul_ir ? "linear_rows_mul_ir" : "linear_rows", stream);
#define FLEX_ARGS(TI) static_cast<const FlexBlock*>(blocks), static_cast<const FlexPart*>(parts), nblocks, column_tiles, static_cast<const TI*>(A), lda, static_cast<const TI*>(W), static_cast<TI*>(C), ldc, rows
#define FLEX(TI)                                                                                                                                                       \
  do {                                                                                                                                                                 \
    if (transposed_weights) {                                                                                                                                          \
      if (shared) hipLaunchKernelGGL((flex_rows_kernel<TI, true, 1, 4>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, FLEX_ARGS(TI));                    \
      else if (big) hipLaunchKernelGGL((flex_rows_kernel<TI, true, 2, 1>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, FLEX_ARGS(TI));                            \
      else hipLaunchKernelGGL((flex_rows_kernel<TI, true, 1, 1>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, FLEX_ARGS(TI));                                \
    } else {                                                                                                                                                           \
      if (shared) hipLaunchKernelGGL((flex_rows_kernel<TI, false, 1, 4>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, FLEX_ARGS(TI));                    \
      else if (big) hipLaunchKernelGGL((flex_rows_kernel<TI, false, 2, 1>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, FLEX_ARGS(TI));                           \
      else hipLaunchKernelGGL((flex_rows_kernel<TI, false, 1, 1>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, FLEX_ARGS(TI));                               \
    }                                                                                                                                                                  \
  } while (0)
  FLEX_DISPATCH(dtype, FLEX);
#undef FLEX
#undef FLEX_ARGS
  CUEQ_CHECK_HIP(hipGetLastError());
  return CUEQ_OK;
}

extern "C" int64_t cueq_linear_flex_dw_chunks(int64_t rows, int32_t tiles) {
  int64_t chunks = 8ll * device_cus() / std::max(1, tiles);  // two wavefronts per SIMD
  // at least 16 rows each: what a chunk of few rows costs is the latency of its chain of loads (64 rows of 9 components: 50 us)
  chunks = std::min<int64_t>(chunks, (rows + 15) / 16);
  return std::max<int64_t>(1, chunks);
}

extern "C" int cueq_linear_flex_dw(int32_t dtype, int64_t rows, const void* X, int64_t ldx, const void* G, int64_t ldg, const void* grads, int32_t ngrads,
                                   int32_t tiles, int64_t numel, float* partial, int32_t mul_ir, int32_t out_dtype, void* dW, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  CUEQ_REQUIRE(dtype == CUEQ_F32 || dtype == CUEQ_BF16 || dtype == CUEQ_F16, CUEQ_ERR_UNSUPPORTED, "linear_flex_dw: dtype must be float32, bfloat16 or half");
  CUEQ_REQUIRE(rows > 0 && ngrads > 0 && tiles > 0 && numel > 0, CUEQ_ERR_INVALID, "linear_flex_dw: bad extents");
  CUEQ_REQUIRE(X && G && grads && partial && dW, CUEQ_ERR_INVALID, "linear_flex_dw: null operand");
  const int64_t chunks = cueq_linear_flex_dw_chunks(rows, tiles);
  const int64_t rpc = ((rows + chunks - 1) / chunks + 15) / 16 * 16, used = (rows + rpc - 1) / rpc;
  const int64_t grid = (used * tiles + 3) / 4;
  CUEQ_REQUIRE(grid < (1ll << 31), CUEQ_ERR_TOO_LARGE, "linear_flex_dw: too many tiles");
  {
    KernelTimer timer(mul_ir ? "linear_dw_mul_ir" : "gemm_tn", stream);
#define FLEX(TI) hipLaunchKernelGGL(flex_grad_kernel<TI>, dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, static_cast<const FlexGrad*>(grads), ngrads, tiles, static_cast<const TI*>(X), ldx, static_cast<const TI*>(G), ldg, partial, numel, rows, rpc, used)
    FLEX_DISPATCH(dtype, FLEX);
#undef FLEX
  }
  CUEQ_CHECK_HIP(hipGetLastError());
#define FLEX(TI) hipLaunchKernelGGL(flex_sum_kernel<TI>, dim3(static_cast<unsigned>((numel + 63) / 64)), dim3(1024), 0, stream, partial, static_cast<TI*>(dW), used, numel)
  FLEX_DISPATCH(out_dtype, FLEX);
#undef FLEX
  CUEQ_CHECK_HIP(hipGetLastError());
  return CUEQ_OK;
}

extern "C" int cueq_sum_runs(const float* partial, int32_t per, int32_t nruns, const int32_t* first, const int64_t* w0, int32_t out_dtype, void* out, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  CUEQ_REQUIRE(partial && first && w0 && out && per > 0 && nruns > 0, CUEQ_ERR_INVALID, "sum_runs: bad arguments");
  CUEQ_REQUIRE(out_dtype == CUEQ_F32 || out_dtype == CUEQ_BF16 || out_dtype == CUEQ_F16, CUEQ_ERR_UNSUPPORTED, "sum_runs: dtype must be float32, bfloat16 or half");
  for (int b0 = 0; b0 < nruns; b0 += 32) {
    const int n = std::min(32, nruns - b0);
    RunTable t;
    for (int b = 0; b < n; ++b) {
      t.first[b] = first[b0 + b];
      t.w0[b] = w0[b0 + b];
    }
    t.first[n] = first[b0 + n];
#define FLEX(TI) hipLaunchKernelGGL(run_sum_kernel<TI>, dim3(static_cast<unsigned>((per + 63) / 64), static_cast<unsigned>(n)), dim3(1024), 0, stream, partial, static_cast<TI*>(out), t, per)
    FLEX_DISPATCH(out_dtype, FLEX);
#undef FLEX
    CUEQ_CHECK_HIP(hipGetLastError());
  }
  return CUEQ_OK;
}
