// Equivariant Linear (uv,iu,iv) for batches that do not fill the chip with the row-streaming kernels (linear_rows*.hip: all
// weights of a launch in LDS, one block per CU, one wavefront per 32 rows and whole column block), and for shapes those do not
// take: any number of input blocks per output block, extents that are multiples of 8 (float) or 16 (2-byte), rows in ir_mul or
// mul_ir.  One launch computes every block of the result, one the partial products of every weight block.
//
//   out[z, c0 + v D + i] = sum over the parts p of the block  coeff_p sum_u A[z, a_p + u D + i] W_p[u, v]
//
// The unit of work is a tile of 32 rows and 32 columns (the row-streaming kernels give a wavefront 32 x 128).  The products are
// issued as W-columns x rows: a lane then holds one row and, per accumulator, 4 adjacent columns of it (times D components in
// mul_ir), both in whole 16-byte pieces; the k order inside a step is free, so a lane takes 4 (8) adjacent channels of its row.
#include <algorithm>
#include <type_traits>

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
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

enum { kFlexMulIr = 1, kFlexOneComponent = 2, kFlexWholePieces = 4 };  // what a caller says of its blocks (cueq_linear_flex's last number)

// The block of a column tile (`tile`: of all blocks, then of its own), nblocks past the last; the whole wavefront is here.  One after the other
// the extents are a chain of loads (16 blocks of an l <= 3 row: 2 us of a kernel of 10), so the lanes read them at once where there are
// more than a few; for three the sums over lanes take longer (0.5 us).
// BACK: the blocks from the last to the first.
template <bool BACK>
__device__ __forceinline__ int flex_find_block(const FlexBlock* __restrict__ blocks, int nblocks, int& tile) {
  if (nblocks <= 6) {
    int b = 0;
    while (b < nblocks && tile >= blocks[BACK ? nblocks - 1 - b : b].nt) tile -= blocks[BACK ? nblocks - 1 - b++ : b++].nt;
    return b;
  }
  const int lane = threadIdx.x & 63;
  for (int first = 0;; first += 64) {
    const int i = first + lane;
    int sum = i < nblocks ? blocks[BACK ? nblocks - 1 - i : i].nt : 1 << 24;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
      const int below = __shfl_up(sum, d, 64);
      sum += lane >= d ? below : 0;
    }
    const int before = __builtin_amdgcn_readfirstlane(__popcll(__ballot(sum <= tile)));
    if (before) tile -= __builtin_amdgcn_readlane(sum, before - 1);
    if (before < 64) return first + before;
  }
}

constexpr int kFlexStageBytes = 2 * 128 * (32 * 7 + 16);  // two buffers of 128 rows x 8 channels (float) x 7 components, the largest

// The weights of a step of the contraction (STEP channels) as the matrix instructions take them, a column of W per lane (WT: a row of
// W, read transposed for the input gradient).  2-byte weights read down a column are a word each until they are used.
template <typename TI, bool WT>
struct FlexWeights {
  static constexpr int ES = sizeof(TI), EPV = 16 / ES, STEP = 2 * EPV;  // channels per step: 4 + 4 (float), 8 + 8
  uint32_t v[WT || ES == 4 ? 4 : 8];
  // lane: this lane's column n and half h: n K + EPV h (WT), EPV h N + n
  static __device__ __forceinline__ uint32_t lane_of(int n, int h, int K, int N) {
    return WT ? static_cast<uint32_t>(n) * K + EPV * h : static_cast<uint32_t>(EPV * h) * N + n;
  }
  __device__ __forceinline__ void load(const TI* __restrict__ w, int k0, int N, uint32_t lane) {
    if constexpr (WT) {
      const uint4 q = *reinterpret_cast<const uint4*>(w + k0 + lane);
      v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    } else {
      using Word = std::conditional_t<ES == 4, uint32_t, uint16_t>;
#pragma unroll
      for (int s = 0; s < EPV; ++s) v[s] = (reinterpret_cast<const Word*>(w) + static_cast<int64_t>(k0 + s) * N)[lane];
    }
  }
  // acc[i] += W x for the D components of the lane's row, x as it lies: EPV channels of D components
  template <int D>
  __device__ __forceinline__ void multiply(const uint4 (&x)[D], fx16 (&acc)[D]) const {
    if constexpr (ES == 4) {
      const float* xf = reinterpret_cast<const float*>(&x[0]);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < D; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(v[s]), xf[s * D + i], acc[i], 0, 0, 0);
    } else {
      uint4 w;
      if constexpr (WT) w = make_uint4(v[0], v[1], v[2], v[3]);
      else w = make_uint4(v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, v[6] | v[7] << 16);
#pragma unroll
      for (int i = 0; i < D; ++i) {
        uint4 op;
        if constexpr (D == 1) op = x[0];
        else op = make_uint4(mm_pick(&x[0], i, D + i), mm_pick(&x[0], 2 * D + i, 3 * D + i), mm_pick(&x[0], 4 * D + i, 5 * D + i), mm_pick(&x[0], 6 * D + i, 7 * D + i));
        acc[i] = mm_32x32x16<TI>(w, op, acc[i]);
      }
    }
  }
};

// what is summed so far counts in units of the coefficient of the part before
template <int D>
__device__ __forceinline__ void flex_rescale(fx16 (&acc)[D], float& scale, float coeff, bool first) {
  if (!first && coeff != scale) {
    const float f = scale / coeff;
#pragma unroll
    for (int i = 0; i < D; ++i) acc[i] *= f;
  }
  scale = coeff;
}

// columns n0 .. n0 + 32 of row z: four adjacent columns of D components at a time
template <typename TI, int D>
__device__ __forceinline__ void flex_store(const FlexBlock& blk, TI* __restrict__ C, int64_t ldc, int64_t z, int n0, int h, const fx16 (&acc)[D], float scale) {
  TI* out = C + z * ldc + blk.c0;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int m = n0 + 8 * a + 4 * h;
    if (m >= blk.N) continue;
    float v[4 * D];
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int i = 0; i < D; ++i) v[b * D + i] = scale * acc[i][4 * a + b];
    if constexpr (sizeof(TI) == 4) {
#pragma unroll
      for (int i = 0; i < D; ++i) *reinterpret_cast<float4*>(out + m * D + 4 * i) = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
    } else {
#pragma unroll
      for (int i = 0; i < D; ++i)
        *reinterpret_cast<uint2*>(out + m * D + 4 * i) = make_uint2(mm_pack<TI>(v[4 * i], v[4 * i + 1]), mm_pack<TI>(v[4 * i + 2], v[4 * i + 3]));
    }
  }
}

// The same through LDS, 64 D bytes of every row at a time, by a wavefront for itself: a lane's own 16-byte pieces are a write request each
// (20 000 rows of 128x0e+128x1o+128x2e in mul_ir, float: 79 us with such stores, 60 without any).
template <int D>
constexpr int kFlexLineBytes = 32 * (64 * D + 16);
// WHOLE: no row of a block ends in half a piece (2-byte elements, N of 4).  What the ends take is 0.5 us of every kernel of 10 that has the code.
template <bool WHOLE, typename TI, int D>
__device__ __forceinline__ void flex_store_lines(const FlexBlock& blk, TI* __restrict__ C, int64_t ldc, int64_t Z, int64_t z0, int n0, const fx16 (&acc)[D],
                                                 float scale, char* lds) {
  constexpr int ES = sizeof(TI), EPV = 16 / ES, COLS = 64 / ES, OS = 64 * D + 16, OP = 4 * D;  // columns a turn; a row's stride and 16-byte pieces in LDS
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
#pragma unroll
  for (int turn = 0; turn < 32 / COLS; ++turn) {
#pragma unroll
    for (int a = 0; a < COLS / 8; ++a) {
      float v[4 * D];
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < D; ++i) v[b * D + i] = scale * acc[i][4 * (turn * (COLS / 8) + a) + b];
      char* to = lds + c * OS + (8 * a + 4 * h) * D * ES;
#pragma unroll
      for (int i = 0; i < D; ++i) {
        if constexpr (ES == 4) *reinterpret_cast<float4*>(to + 16 * i) = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
        else *reinterpret_cast<uint2*>(to + 8 * i) = make_uint2(mm_pack<TI>(v[4 * i], v[4 * i + 1]), mm_pack<TI>(v[4 * i + 2], v[4 * i + 3]));
      }
    }
    __builtin_amdgcn_wave_barrier();
    const int from_col = (n0 + turn * COLS) * D, ends_col = blk.N * D;
#pragma unroll
    for (int j = 0; j < 2 * D; ++j) {
      const int piece = j * 64 + lane, r = piece / OP, q = piece % OP;
      const int64_t z = z0 + r;
      const u32x4 value = *reinterpret_cast<const u32x4*>(lds + r * OS + 16 * q);
      if (z < Z && from_col + (WHOLE ? q * EPV : q * EPV + EPV - 1) < ends_col) *reinterpret_cast<u32x4*>(C + z * ldc + blk.c0 + from_col + q * EPV) = value;
    }
    if constexpr (!WHOLE) {
      const int half = ends_col - 4 - from_col;
      if (ends_col % EPV && half >= 0 && half < COLS * D && h == 0 && z0 + c < Z)
        *reinterpret_cast<uint2*>(C + (z0 + c) * ldc + blk.c0 + from_col + half) = *reinterpret_cast<const uint2*>(lds + c * OS + half * ES);
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// ---- few tiles: the four wavefronts of a workgroup share a tile of 32 rows and 32 columns, each with its part of every contraction;
// the first adds the others' sums, in order, through LDS and stores.  A lane reads its own row; the operands of PD steps are in
// flight, as many as the registers beside the sums allow.
template <typename TI, int D, bool WT>
__device__ __forceinline__ void flex_shared_tile(const FlexBlock& blk, const FlexPart* __restrict__ parts, const TI* __restrict__ A, int64_t lda,
                                                 const TI* __restrict__ W, TI* __restrict__ C, int64_t ldc, int64_t Z, int64_t z0, int n0) {
  using Weights = FlexWeights<TI, WT>;
  constexpr int EPV = Weights::EPV, STEP = Weights::STEP, PD = D == 1 ? 8 : D == 3 || (D == 5 && (WT || sizeof(TI) == 4)) ? 4 : 2;
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int share = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  fx16 acc[D];
#pragma unroll
  for (int i = 0; i < D; ++i) acc[i] = fx16{0};
  const int n = min(n0 + c, blk.N - 1);
  const TI* row = A + min(z0 + c, Z - 1) * lda;
  float scale = 1.0f;
  for (int p = 0; p < blk.parts; ++p) {
    const FlexPart part = parts[blk.first + p];
    flex_rescale(acc, scale, part.coeff, p == 0);
    const int steps = part.K / STEP, first = steps * share / 4 * STEP, last = steps * (share + 1) / 4 * STEP;
    if (first == last) continue;
    uint4 x[PD][D];
    Weights w[PD];
    const uint32_t w_lane = Weights::lane_of(n, h, part.K, blk.N);
    auto load = [&](int k0, uint4 (&xx)[D], Weights& ww) {
#pragma unroll
      for (int i = 0; i < D; ++i) xx[i] = *reinterpret_cast<const uint4*>(row + part.a0 + static_cast<int64_t>(k0 + EPV * h) * D + i * EPV);
      ww.load(W + part.w0, k0, blk.N, w_lane);
    };
#pragma unroll
    for (int j = 0; j < PD; ++j)
      if (first + j * STEP < last) load(first + j * STEP, x[j], w[j]);
    for (int k0 = first; k0 < last; k0 += PD * STEP)
#pragma unroll
      for (int j = 0; j < PD; ++j) {
        if (k0 + j * STEP < last) {
          w[j].multiply(x[j], acc);
          if (k0 + (PD + j) * STEP < last) load(k0 + (PD + j) * STEP, x[j], w[j]);
        }
      }
  }
  __shared__ float others[3][16][64];
#pragma unroll
  for (int i = 0; i < D; ++i) {
    if (share)
#pragma unroll
      for (int r = 0; r < 16; ++r) others[share - 1][r][lane] = acc[i][r];
    __syncthreads();
    if (!share)
#pragma unroll
      for (int r = 0; r < 16; ++r)
#pragma unroll
        for (int o = 0; o < 3; ++o) acc[i][r] += others[o][r][lane];
    __syncthreads();
  }
  if (share == 0 && z0 + c < Z) flex_store(blk, C, ldc, z0 + c, n0, h, acc, scale);
}

// unit = (column tiles of the blocks one after the other) x (row tile)
template <typename TI, bool WT>
__global__ void __launch_bounds__(256, 2) flex_shared_kernel(const FlexBlock* __restrict__ blocks, const FlexPart* __restrict__ parts, int nblocks, int tiles_n,
                                                             const TI* __restrict__ A, int64_t lda, const TI* __restrict__ W, TI* __restrict__ C, int64_t ldc,
                                                             int64_t Z) {
  const uint32_t column = static_cast<uint32_t>(tiles_n), zt = blockIdx.x / column;
  const int64_t z0 = static_cast<int64_t>(zt) * 32;
  int tile = static_cast<int>(blockIdx.x - zt * column);
  const int b = flex_find_block<false>(blocks, nblocks, tile);
  if (b >= nblocks || z0 >= Z) return;
  const FlexBlock blk = blocks[b];
  switch (blk.D) {
    case 1: flex_shared_tile<TI, 1, WT>(blk, parts, A, lda, W, C, ldc, Z, z0, tile * 32); break;
    case 3: flex_shared_tile<TI, 3, WT>(blk, parts, A, lda, W, C, ldc, Z, z0, tile * 32); break;
    case 5: flex_shared_tile<TI, 5, WT>(blk, parts, A, lda, W, C, ldc, Z, z0, tile * 32); break;
    default: flex_shared_tile<TI, 7, WT>(blk, parts, A, lda, W, C, ldc, Z, z0, tile * 32);
  }
}

// ---- blocks of few columns: a wavefront has ZT row tiles and a column tile to itself; the operands of two steps are in flight, and a lane
// reads its own rows, whose lines the next steps and the neighbouring column tiles find in L1.  Bound by the latency of a tile's few
// steps, so by how many wavefronts a SIMD holds (more steps in flight cost registers, and 1.05 to 1.3 times as long); the result leaves in
// lines.  A workgroup that stages rows for one or two column tiles reads half or a quarter of a line of every row and step and
// waits for all four wavefronts.  Forward of 0e+1o+2e rows in ir_mul, us, staged / this: float 16 ch 20 000 rows 17 / 9.7, 64 ch 9 000
// 19.5 / 16.3, 96 ch 4 500 22.4 / 17.7; bfloat16 16 ch 20 000 15.3 / 7.3, 96 ch 4 500 14.6 / 10.6, l <= 3 48 ch 9 000 22.7 / 13.0.
template <typename TI, int D, int ZT, bool WT>
__device__ __forceinline__ void flex_direct_tile(const FlexBlock& blk, const FlexPart* __restrict__ parts, const TI* __restrict__ A, int64_t lda,
                                                 const TI* __restrict__ W, TI* __restrict__ C, int64_t ldc, int64_t Z, int64_t z0, int n0, char* lds) {
  using Weights = FlexWeights<TI, WT>;
  constexpr int EPV = Weights::EPV, STEP = Weights::STEP, PD = 2;
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
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
#pragma unroll
    for (int t = 0; t < ZT; ++t) {
      float before = scale;
      flex_rescale(acc[t], before, part.coeff, p == 0);
    }
    scale = part.coeff;
    const int K = part.K;
    uint4 x[PD][ZT][D];
    Weights w[PD];
    const uint32_t w_lane = Weights::lane_of(n, h, K, blk.N);
    auto load = [&](int k0, uint4 (&xx)[ZT][D], Weights& ww) {  // (past the end the last step again: not used)
      const int k = min(k0, K - STEP);
#pragma unroll
      for (int t = 0; t < ZT; ++t)
#pragma unroll
        for (int i = 0; i < D; ++i) xx[t][i] = *reinterpret_cast<const uint4*>(row[t] + part.a0 + static_cast<int64_t>(k + EPV * h) * D + i * EPV);
      ww.load(W + part.w0, k, blk.N, w_lane);
    };
#pragma unroll
    for (int j = 0; j < PD; ++j) load(j * STEP, x[j], w[j]);
    int k0 = 0;
    for (; k0 + PD * STEP <= K; k0 += PD * STEP)
#pragma unroll
      for (int j = 0; j < PD; ++j) {
#pragma unroll
        for (int t = 0; t < ZT; ++t) w[j].multiply(x[j][t], acc[t]);
        load(k0 + (PD + j) * STEP, x[j], w[j]);
      }
#pragma unroll
    for (int j = 0; j < PD - 1; ++j)
      if (k0 + j * STEP < K)
#pragma unroll
        for (int t = 0; t < ZT; ++t) w[j].multiply(x[j][t], acc[t]);
  }
#pragma unroll
  for (int t = 0; t < ZT; ++t) flex_store_lines<true>(blk, C, ldc, Z, z0 + 32 * t, n0, acc[t], scale, lds);
}

// unit = (column tiles of the blocks one after the other) x (ZT row tiles), four to a workgroup: its wavefronts share rows.  ONE: every
// block has one component.
template <typename TI, bool WT, bool ONE, int ZT>
__global__ void __launch_bounds__(256, ONE ? (ZT == 1 ? 4 : 3) : 2) flex_direct_kernel(const FlexBlock* __restrict__ blocks, const FlexPart* __restrict__ parts, int nblocks,
                                                                                      int tiles_n, const TI* __restrict__ A, int64_t lda, const TI* __restrict__ W,
                                                                                      TI* __restrict__ C, int64_t ldc, int64_t Z) {
  __shared__ __align__(16) char lines[4][ONE ? kFlexLineBytes<1> : kFlexLineBytes<7>];
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const uint32_t column = static_cast<uint32_t>(tiles_n), unit = blockIdx.x * 4 + wave, zt = unit / column;  // (grid x 4 < 2^32)
  const int64_t z0 = static_cast<int64_t>(zt) * (32 * ZT);
  int tile = static_cast<int>(unit - zt * column);
  const int b = flex_find_block<false>(blocks, nblocks, tile);
  if (b >= nblocks || z0 >= Z) return;
  const FlexBlock blk = blocks[b];
  char* lds = lines[wave];
  if constexpr (ONE) {
    flex_direct_tile<TI, 1, ZT, WT>(blk, parts, A, lda, W, C, ldc, Z, z0, tile * 32, lds);
  } else {
    switch (blk.D) {
      case 1: flex_direct_tile<TI, 1, ZT, WT>(blk, parts, A, lda, W, C, ldc, Z, z0, tile * 32, lds); break;
      case 3: flex_direct_tile<TI, 3, ZT, WT>(blk, parts, A, lda, W, C, ldc, Z, z0, tile * 32, lds); break;
      case 5: flex_direct_tile<TI, 5, ZT, WT>(blk, parts, A, lda, W, C, ldc, Z, z0, tile * 32, lds); break;
      default: flex_direct_tile<TI, 7, ZT, WT>(blk, parts, A, lda, W, C, ldc, Z, z0, tile * 32, lds);
    }
  }
}

// ---- more tiles: a workgroup stages its rows through LDS.  Bound by the matrix cores from some 10 000 rows of float on (20 000 rows of
// 128x0e+128x1o+128x2e in mul_ir, forward: 131 -> 73 us, 80 TFLOP/s; 38 at the rate of a large product), below by the latency of the
// first and last step of a tile (5 003 rows 37 -> 24 us), in 2-byte elements by bytes and latency (8 000 rows 25 -> 13 us).
// A workgroup has RT row tiles of 32 and 4 / RT column tiles of a block, a wavefront each one of the four pairs (MIXED, RT = 2: three have
// the row tile at z0, the fourth that at z1 and a column tile of its own).  The rows come in
// chunks of 4 / RT steps, two buffers in turn, one barrier a chunk: 128 D / RT adjacent bytes of every row, whole lines of
// memory where a lane's own row would be a line per lane and load (64 lines an instruction, four times over for the four
// wavefronts).  16 bytes of padding per row put the lanes' reads on all banks.  The weights go straight to registers, four steps ahead.
template <typename TI, int D, int RT, int ZT, bool WT, bool WHOLE, bool MIXED = false>
__device__ __forceinline__ void flex_stage_tile(const FlexBlock& blk, const FlexPart* __restrict__ parts, const TI* __restrict__ A, int64_t lda,
                                                const TI* __restrict__ W, TI* __restrict__ C, int64_t ldc, int64_t Z, int64_t z0, int first_tile, char* lds, int64_t z1 = 0, int last_tile = 0) {
  using Weights = FlexWeights<TI, WT>;
  constexpr int ES = sizeof(TI), EPV = Weights::EPV, STEP = Weights::STEP;
  constexpr int SPC = 4 / RT, KC = SPC * STEP;                       // steps and channels of a chunk
  constexpr int PR = KC * D * ES / 16, RS = PR * 16 + 16, BUF = 32 * RT * ZT * RS;  // 16-byte pieces of a row, its stride, a buffer
  constexpr int NP = D * ZT;                                                        // pieces a lane brings
  static_assert(32 * RT * ZT * PR == 256 * NP && 2 * BUF <= kFlexStageBytes, "the rows of a chunk");
  static_assert(4 * kFlexLineBytes<D> <= kFlexStageBytes, "the lines of four wavefronts");
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int rt = MIXED ? wave == 3 : wave / (4 / RT), n0 = 32 * (!MIXED ? first_tile + wave % (4 / RT) : rt ? last_tile : first_tile + wave);
  fx16 acc[ZT][D];
#pragma unroll
  for (int t = 0; t < ZT; ++t)
#pragma unroll
    for (int i = 0; i < D; ++i) acc[t][i] = fx16{0};
  const int n = min(n0 + c, blk.N - 1);
  const TI* from[NP];  // this lane's pieces of a chunk
  int into[NP], col[NP];
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    const int piece = j * 256 + threadIdx.x, r = piece / PR, q = piece % PR;
    from[j] = A + min(MIXED && r >= 32 * ZT ? z1 + (r - 32 * ZT) : z0 + r, Z - 1) * lda;
    into[j] = r * RS + q * 16;
    col[j] = q * EPV;
  }
  const char* mine = lds + (32 * rt * ZT + c) * RS + EPV * h * D * ES;
  float scale = 1.0f;
  int turn = 0;
  for (int p = 0; p < blk.parts; ++p) {
    const FlexPart part = parts[blk.first + p];
#pragma unroll
    for (int t = 0; t < ZT; ++t) {
      float before = scale;
      flex_rescale(acc[t], before, part.coeff, p == 0);
    }
    scale = part.coeff;
    const int K = part.K, ends = K * D - EPV;  // (pieces past the row's channels repeat its last one and are not used)
    u32x4 x[NP];  // (a vector type: an array of structs stays in memory here)
    auto fetch = [&](int k0) {
#pragma unroll
      for (int j = 0; j < NP; ++j) x[j] = *reinterpret_cast<const u32x4*>(from[j] + part.a0 + min(k0 * D + col[j], ends));
    };
    constexpr int WD = D == 7 && ES == 2 ? 2 : 4;  // (as the registers allow)
    Weights w[WD];
    const uint32_t w_lane = Weights::lane_of(n, h, K, blk.N);
    fetch(0);
#pragma unroll
    for (int s = 0; s < WD; ++s) w[s].load(W + part.w0, min(s * STEP, K - STEP), blk.N, w_lane);
    // (whole groups of four steps without a condition: behind one the number of loads on the way is unknown, and every wait is for
    // all of them)
    auto four = [&](int k4, auto whole) {
#pragma unroll
      for (int ch = 0; ch < RT; ++ch) {
        const int k0 = k4 + ch * KC;
        if (!decltype(whole)::value && k0 >= K) continue;
        char* buf = lds + turn * BUF;
#pragma unroll
        for (int j = 0; j < NP; ++j) *reinterpret_cast<u32x4*>(buf + into[j]) = x[j];
        __syncthreads();  // (the other buffer is no longer read once every wavefront is here)
        fetch(k0 + KC);
#pragma unroll
        for (int s = 0; s < SPC; ++s) {
          const int k = k0 + s * STEP;
          if (!decltype(whole)::value && k >= K) continue;
#pragma unroll
          for (int t = 0; t < ZT; ++t) {
            uint4 op[D];
            if constexpr (D == 7 && ES == 2 && WT) __builtin_amdgcn_sched_barrier(0);  // (a step at a time: 54 registers spilled, so 4)
#pragma unroll
            for (int i = 0; i < D; ++i) op[i] = *reinterpret_cast<const uint4*>(mine + turn * BUF + 32 * t * RS + s * STEP * D * ES + 16 * i);
            w[(ch * SPC + s) % WD].multiply(op, acc[t]);
          }
          w[(ch * SPC + s) % WD].load(W + part.w0, min(k + WD * STEP, K - STEP), blk.N, w_lane);
        }
        turn ^= 1;
      }
    };
    int k4 = 0;
    for (; k4 + 4 * STEP <= K; k4 += 4 * STEP) four(k4, std::true_type{});
    if (k4 < K) four(k4, std::false_type{});
  }
  __syncthreads();  // (no wavefront reads the rows any more)
#pragma unroll
  for (int t = 0; t < ZT; ++t) flex_store_lines<WHOLE>(blk, C, ldc, Z, (MIXED && rt ? z1 : z0 + 32 * ZT * rt) + 32 * t, n0, acc[t], scale, lds + wave * kFlexLineBytes<D>);
}

// A slab of 128 ZT rows and a block of nt column tiles are nt workgroups: four columns x one row tile for every whole four columns.  Of
// those that are left, one is four row tiles, two are two x two, and three are three workgroups of three columns x one row tile and,
// by the fourth wavefront, one column of the last row tile (as three x four row tiles, rows staged three times over, 96 ch took twice
// as long).  The last block first: the blocks of most components are the longest.  ZT > 1: row
// tiles of a wavefront, where every block has one component (a tile of one is over before its first loads have paid).
template <typename TI, bool WT, int ZT, bool WHOLE>
__global__ void __launch_bounds__(256, 2) flex_stage_kernel(const FlexBlock* __restrict__ blocks, const FlexPart* __restrict__ parts, int nblocks,
                                                            const TI* __restrict__ A, int64_t lda, const TI* __restrict__ W, TI* __restrict__ C, int64_t ldc,
                                                            int64_t Z, int64_t slabs) {
  __shared__ __align__(16) char lds[kFlexStageBytes];
  const uint32_t column = blockIdx.x / static_cast<uint32_t>(slabs);  // (slab and column tile of a block run over slabs x its extent)
  int before = static_cast<int>(column);
  const int b = nblocks - 1 - flex_find_block<true>(blocks, nblocks, before);
  if (b < 0) return;
  const FlexBlock blk = blocks[b];
  const uint32_t own = blockIdx.x - static_cast<uint32_t>(slabs) * (column - before), slab = own / static_cast<uint32_t>(blk.nt);
  const int t = static_cast<int>(own - slab * blk.nt), full = blk.nt & ~3, rest = blk.nt - full;
  const int64_t zs = static_cast<int64_t>(slab) * (128 * ZT);
  constexpr int RZ = 32 * ZT;  // rows of a row tile
#define STAGE(D)                                                                                                              \
  do {                                                                                                                       \
    if (t < full) {                                                                                                          \
      const int64_t z0 = zs + (t & 3) * RZ;                                                                                   \
      if (z0 < Z) flex_stage_tile<TI, D, 1, ZT, WT, WHOLE>(blk, parts, A, lda, W, C, ldc, Z, z0, t & ~3, lds);                  \
    } else if (rest == 1) {                                                                                                  \
      if (zs < Z) flex_stage_tile<TI, D, 4, ZT, WT, WHOLE>(blk, parts, A, lda, W, C, ldc, Z, zs, full, lds);                    \
    } else if (rest == 2) {                                                                                                  \
      const int64_t z0 = zs + 2 * (t - full) * RZ;                                                                            \
      if (z0 < Z) flex_stage_tile<TI, D, 2, ZT, WT, WHOLE>(blk, parts, A, lda, W, C, ldc, Z, z0, full, lds);                    \
    } else {                                                                                                                 \
      const int64_t z0 = zs + (t - full) * RZ;                                                                                \
      if (z0 < Z) flex_stage_tile<TI, D, 2, ZT, WT, WHOLE, true>(blk, parts, A, lda, W, C, ldc, Z, z0, full, lds, zs + 3 * RZ, t); \
    }                                                                                                                        \
  } while (0)
  if constexpr (ZT > 1) {
    STAGE(1);
  } else {
    switch (blk.D) {
      case 1: STAGE(1); break;
      case 3: STAGE(3); break;
      case 5: STAGE(5); break;
      default: STAGE(7);
    }
  }
#undef STAGE
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
  // four wavefronts share a tile where all tiles, four wavefronts each, still run at once (two workgroups to a CU): 300 rows of
  // 128x0e+128x1o+128x2e in mul_ir, float, forward 21.8 -> 9.7 us, 1 000 rows 22.1 -> 12.6 (1 400 rows, past the line: 22.5 either way)
  const int64_t tiles = (rows + 31) / 32 * column_tiles;
  const bool shared = tiles <= 2ll * device_cus();
  // Rows in ir_mul (the caller says that every block has one component).  Four staged row tiles a wavefront once there are so many
  // workgroups; us for one / four, 128 ch l <= 2: float 4 000 rows (1 152 workgroups of one tile) 23 / 26, 8 000 38 / 38, 16 000 67 / 57,
  // 32 000 147 / 113; bfloat16 2 000 9.8 / 9.7, 4 000 13.8 / 9.8, 32 000 73 / 35.  One where the columns are whole groups of four (or four
  // and two: 192 ch, float, 1 000 rows 16 / 16.6, 3 000 53 / 51, so staged up to some 5 000 tiles).  Otherwise a wavefront has its tile to
  // itself, and two row tiles from three column tiles a block on (their weights are read half as often: us for one / two, 96 ch l <= 2, float, input
  // gradient 9 000 rows 34 / 29, bfloat16 9 000 18.6 / 16.0; 64 ch, float, forward 9 000 16.3 / 18.1).
  // Rows in mul_ir: a component more is a longer step, and staging is the faster way but for one column tile of 2-byte elements
  // and few rows (16 ch l <= 2, 6 500 rows, 7.6 / 7.0; 32 ch l <= 3, 20 000 13.3 / 16.0).
  const bool whole = dtype == CUEQ_F32 || (mul_ir & kFlexWholePieces), one = (mul_ir & kFlexOneComponent) && whole;
  const bool tall = one && !shared && column_tiles >= (dtype == CUEQ_F32 ? 4 : 3) * nblocks &&
                    (rows + 127) / 128 * column_tiles >= (dtype == CUEQ_F32 ? 9ll : 4ll) * device_cus();
  const bool even = column_tiles >= 4 * nblocks && column_tiles % (2 * nblocks) == 0;  // (on average: blocks of groups of four and two columns)
  const bool direct = whole && !shared && !tall && (one ? !even || (dtype == CUEQ_F32 && column_tiles % (4 * nblocks) != 0 && tiles > 20ll * device_cus())
                                                         : dtype != CUEQ_F32 && column_tiles == nblocks && tiles <= 4ll * device_cus());
  const int zt = one && column_tiles >= 3 * nblocks && tiles >= 16ll * device_cus() ? 2 : 1;
  const int64_t slab_rows = tall ? 512 : 128, slabs = (rows + slab_rows - 1) / slab_rows;
  const int64_t grid = shared ? tiles : direct ? ((rows + 32 * zt - 1) / (32 * zt) * column_tiles + 3) / 4 : slabs * column_tiles;
  CUEQ_REQUIRE(grid < (1ll << 30), CUEQ_ERR_TOO_LARGE, "linear_flex: too many rows");
  KernelTimer timer(mul_ir & kFlexMulIr ? "linear_rows_mul_ir" : "linear_rows", stream);
#define FLEX_LAUNCH(KERNEL, ...)                                                                                                                         \
  hipLaunchKernelGGL((KERNEL), dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, static_cast<const FlexBlock*>(blocks),                           \
                     static_cast<const FlexPart*>(parts), nblocks, __VA_ARGS__)
#define FLEX_OPERANDS(TI) static_cast<const TI*>(A), lda, static_cast<const TI*>(W), static_cast<TI*>(C), ldc, rows
#define FLEX_WT(TI, WT)                                                                                                    \
  do {                                                                                                                      \
    if (shared) FLEX_LAUNCH((flex_shared_kernel<TI, WT>), column_tiles, FLEX_OPERANDS(TI));                                   \
    else if (direct && !one) FLEX_LAUNCH((flex_direct_kernel<TI, WT, false, 1>), column_tiles, FLEX_OPERANDS(TI));         \
    else if (direct && zt == 1) FLEX_LAUNCH((flex_direct_kernel<TI, WT, true, 1>), column_tiles, FLEX_OPERANDS(TI));       \
    else if (direct) FLEX_LAUNCH((flex_direct_kernel<TI, WT, true, 2>), column_tiles, FLEX_OPERANDS(TI));                  \
    else if (tall) FLEX_LAUNCH((flex_stage_kernel<TI, WT, 4, true>), FLEX_OPERANDS(TI), slabs);                               \
    else if (whole || sizeof(TI) == 4) FLEX_LAUNCH((flex_stage_kernel<TI, WT, 1, true>), FLEX_OPERANDS(TI), slabs);           \
    else FLEX_LAUNCH((flex_stage_kernel<TI, WT, 1, sizeof(TI) == 4>), FLEX_OPERANDS(TI), slabs);                              \
  } while (0)
#define FLEX(TI) do { if (transposed_weights) FLEX_WT(TI, true); else FLEX_WT(TI, false); } while (0)
  FLEX_DISPATCH(dtype, FLEX);
#undef FLEX
#undef FLEX_WT
#undef FLEX_OPERANDS
#undef FLEX_LAUNCH
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
