// Operations that scale every row of a tensor by one number of that row.
#include "common.h"
#include "cw_common.h"
#include "u1d_spec.h"

namespace cueq {
namespace {

template <int DT> struct element;
template <> struct element<CUEQ_F32> { using type = float; };
template <> struct element<CUEQ_F64> { using type = double; };
template <> struct element<CUEQ_F16> { using type = f16_t; };
template <> struct element<CUEQ_BF16> { using type = bf16_t; };

// out[r, :] = in[r, :] / (how many batch rows the grouping puts on row r, at least 1): a block per row, one pass over memory.  A
// layer's mean over its messages took ten launches and two waits of the host to count the degrees that the grouping of the
// product before it holds already: forward + backward of the convolution, fp32, 64 ch, 12 007 edges 706 -> 588 us, 32 ch, 5 000 edges
// 204 -> 102; forward, 64 ch, 300 edges 96 -> 26.
template <typename T>
__global__ void __launch_bounds__(256) rows_mean_kernel(const T* __restrict__ in, const int64_t* __restrict__ offsets, int64_t width, T* __restrict__ out) {
  using M = typename math_of<T>::type;
  const int64_t r = blockIdx.x;
  const int64_t count = offsets[r + 1] - offsets[r];
  const M n = static_cast<M>(count > 1 ? count : 1);
  for (int64_t c = threadIdx.x; c < width; c += blockDim.x) io_st(io_ld(in + r * width + c) / n, out + r * width + c);
}

// 3-vectors divided by their length, n = max(|x|, eps), and the derivatives force training needs; a lane per vector.  PyTorch's
// element-wise kernels took 3 launches for the quotient, 10 for its gradient and 18 for the gradient of that, each a few us for
// a few thousand vectors and more on the host (a force-training step of one layer, 9 001 edges 569 -> 378 us, 1 352 edges
// 599 -> 382).  The gradient goes through |x| where |x| >= eps, as that of a clamp does.
//   STAGE 0: y = x / n
//   STAGE 1: dx = (g - (y.g) y) / n
//   STAGE 2, of v . dx: dg = (v - (y.v) y) / n, dx = (3 (y.v) (y.g) y - (v.g) y - (y.g) v - (y.v) g) / n^2
// Computed in float64 and rounded once: the second derivative cancels (2-norm error over 200 000 random vectors, in float32
// 1.5e-7, so 2.5e-8, PyTorch's operations 5e-8 to 9e-8), and the arithmetic is hidden behind the latency of the loads.
template <typename T, int STAGE>
__global__ void __launch_bounds__(64) normalize3_kernel(const T* __restrict__ x, const T* __restrict__ g, const T* __restrict__ v, int64_t rows, double eps,
                                                        T* __restrict__ out, T* __restrict__ out_x) {
  const int64_t r = static_cast<int64_t>(blockIdx.x) * 64 + threadIdx.x;
  if (r >= rows) return;
  double p[3], n2 = 0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    p[a] = x[3 * r + a];
    n2 = fma(p[a], p[a], n2);
  }
  const double length = sqrt(n2), n = length < eps ? eps : length;
  if constexpr (STAGE == 0) {
#pragma unroll
    for (int a = 0; a < 3; ++a) out[3 * r + a] = static_cast<T>(p[a] / n);
  } else {
    double q[3], y[3], yq = 0;  // q: g (stage 1) or v (stage 2)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      q[a] = (STAGE == 1 ? g : v)[3 * r + a];
      y[a] = p[a] / n;
      yq = fma(y[a], q[a], yq);
    }
    const bool through = !(length < eps);  // (a NaN stays one)
    if (out)
#pragma unroll
      for (int a = 0; a < 3; ++a) out[3 * r + a] = static_cast<T>((q[a] - (through ? yq * y[a] : 0.0)) / n);
    if constexpr (STAGE == 2) {
      if (out_x) {
        double yg = 0, qg = 0, w[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          w[a] = g[3 * r + a];
          yg = fma(y[a], w[a], yg);
          qg = fma(q[a], w[a], qg);
        }
        const double c = 3 * yq * yg - qg;
#pragma unroll
        for (int a = 0; a < 3; ++a) out_x[3 * r + a] = static_cast<T>(through ? (c * y[a] - yg * q[a] - yq * w[a]) / n / n : 0.0);
      }
    }
  }
}

}  // namespace
}  // namespace cueq

using namespace cueq;

#define BY_TYPE(dtype, F)                        \
  switch (dtype) {                               \
    case CUEQ_F32: F(CUEQ_F32); break;           \
    case CUEQ_F64: F(CUEQ_F64); break;           \
    case CUEQ_F16: F(CUEQ_F16); break;           \
    default: F(CUEQ_BF16); break;                \
  }

extern "C" int cueq_rows_mean(int32_t dtype, int64_t rows, int64_t width, const void* in, const int64_t* offsets, void* out, void* stream_) {
  CUEQ_REQUIRE(dtype == CUEQ_F32 || dtype == CUEQ_F64 || dtype == CUEQ_F16 || dtype == CUEQ_BF16, CUEQ_ERR_UNSUPPORTED, "rows_mean: unknown element type");
  CUEQ_REQUIRE(rows >= 0 && width >= 0, CUEQ_ERR_INVALID, "rows_mean: bad extents");
  CUEQ_REQUIRE(rows < (int64_t(1) << 31), CUEQ_ERR_TOO_LARGE, "rows_mean: too many rows for one launch");
  if (rows == 0 || width == 0) return CUEQ_OK;
  CUEQ_REQUIRE(in && offsets && out, CUEQ_ERR_INVALID, "rows_mean: null operand");
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  const unsigned threads = width > 128 ? 256u : width > 64 ? 128u : 64u;
#define MEAN(DT) { using T = element<DT>::type; hipLaunchKernelGGL(rows_mean_kernel<T>, dim3(static_cast<unsigned>(rows)), dim3(threads), 0, stream, static_cast<const T*>(in), offsets, width, static_cast<T*>(out)); }
  BY_TYPE(dtype, MEAN)
#undef MEAN
  CUEQ_CHECK_HIP(hipGetLastError());
  return CUEQ_OK;
}

extern "C" int cueq_normalize3(int32_t dtype, int32_t stage, int64_t rows, const void* x, const void* g, const void* v, double eps, void* out, void* out_x,
                               void* stream_) {
  CUEQ_REQUIRE(dtype == CUEQ_F32 || dtype == CUEQ_F64, CUEQ_ERR_UNSUPPORTED, "normalize3: dtype must be float32 or float64");
  CUEQ_REQUIRE(stage >= 0 && stage <= 2 && rows >= 0, CUEQ_ERR_INVALID, "normalize3: bad arguments");
  const int64_t grid = (rows + 63) / 64;
  CUEQ_REQUIRE(grid < (int64_t(1) << 31), CUEQ_ERR_TOO_LARGE, "normalize3: too many rows for one launch");
  if (rows == 0) return CUEQ_OK;
  CUEQ_REQUIRE(x && (stage < 1 || g) && (stage < 2 || v) && (out || (stage == 2 && out_x)), CUEQ_ERR_INVALID, "normalize3: null operand");
  hipStream_t stream = static_cast<hipStream_t>(stream_);
#define NORMALIZE(T, S) hipLaunchKernelGGL((normalize3_kernel<T, S>), dim3(static_cast<unsigned>(grid)), dim3(64), 0, stream, static_cast<const T*>(x), static_cast<const T*>(g), static_cast<const T*>(v), rows, eps, static_cast<T*>(out), static_cast<T*>(out_x))
#define STAGES(T) do { if (stage == 0) NORMALIZE(T, 0); else if (stage == 1) NORMALIZE(T, 1); else NORMALIZE(T, 2); } while (0)
  if (dtype == CUEQ_F64) STAGES(double);
  else STAGES(float);
#undef STAGES
#undef NORMALIZE
  CUEQ_CHECK_HIP(hipGetLastError());
  return CUEQ_OK;
}
