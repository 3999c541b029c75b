// fp16 / fp32 activations of the fused GEMM as two bf16 terms.
//
// The reference multiplies activations of any type with tl.dot
// (bf16x_gemm_fused.py:89-91).  Here x = hi + lo with hi = bf16(x), lo =
// bf16(x - hi): exact for fp16, 16 significant bits for fp32.  The terms are
// written as 2 M rows of one bf16 matrix, so one GEMM launch decodes the weight
// once for both, and the two halves of its fp32 result are added and rounded
// to x's type.  (Where in_f % 256 == 0, from 33 rows, or 17 of a weight of 2^25
// elements, the wave-specialised GEMM takes both terms itself:
// bf16x_gemm_terms.)  Both kernels are bound by the launch at the sizes they run
// at (64x4096: 2-3 us each); they replace five elementwise passes and a second
// GEMM (3000x4160 fp16 M = 64: 67.6 -> 32.5 us for the call).
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include "../../include/bf16x_hip.h"
#include "bf16x_device.h"
#include "launch_common.h"

namespace {
using namespace bf16x;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float widen(_Float16 v) { return (float)v; }
__device__ __forceinline__ float widen(float v) { return v; }

__device__ __forceinline__ void split1(float f, uint32_t& hi, uint32_t& lo) {
  hi = f32_to_bf16_rne(f);
  lo = f32_to_bf16_rne(f - __uint_as_float(hi << 16));
}

// four elements per thread when VEC (x aligned to four elements, hi and lo to
// 8 bytes), the remainder and the rest one by one
template <typename T, typename V, bool VEC>
__global__ __launch_bounds__(256) void split_kernel(const T* __restrict__ x, int64_t n, uint16_t* __restrict__ hi,
                                                    uint16_t* __restrict__ lo) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  const int64_t n4 = VEC ? n / 4 : 0;
  for (int64_t i = t; i < n4; i += step) {
    const V v = ((const V*)x)[i];
    const T e[4] = {v.x, v.y, v.z, v.w};
    uint32_t h[4], l[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) split1(widen(e[k]), h[k], l[k]);
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    ((u32x2*)hi)[i] = u32x2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
    ((u32x2*)lo)[i] = u32x2{l[0] | (l[1] << 16), l[2] | (l[3] << 16)};
  }
  for (int64_t i = 4 * n4 + t; i < n; i += step) {
    uint32_t h, l;
    split1(widen(x[i]), h, l);
    hi[i] = (uint16_t)h;
    lo[i] = (uint16_t)l;
  }
}

template <typename T, typename V, bool VEC>
__global__ __launch_bounds__(256) void add_kernel(const float* __restrict__ a, const float* __restrict__ b, int64_t n,
                                                  T* __restrict__ y) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  const int64_t n4 = VEC ? n / 4 : 0;
  for (int64_t i = t; i < n4; i += step) {
    const f32x4 s = ((const f32x4*)a)[i] + ((const f32x4*)b)[i];
    ((V*)y)[i] = V{(T)s.x, (T)s.y, (T)s.z, (T)s.w};
  }
  for (int64_t i = 4 * n4 + t; i < n; i += step) y[i] = (T)(a[i] + b[i]);
}

unsigned grid_of(int64_t n) { return (unsigned)std::min<int64_t>((n / 4 + 256) / 256, 8192); }

}  // namespace

extern "C" int bf16x_split_terms(const void* x, int32_t x_dtype, int64_t n, uint16_t* hi, uint16_t* lo,
                                 bf16x_stream_t stream) {
  if (!x || !hi || !lo || n <= 0) return BF16X_EARG;
  if (!aligned2(hi) || !aligned2(lo)) return BF16X_EARG;
  hipStream_t st = (hipStream_t)stream;
  const dim3 g(grid_of(n)), b(256);
  const bool out8 = aligned8(hi) && aligned8(lo);
  if (x_dtype == BF16X_F16) {
    if (!aligned2(x)) return BF16X_EARG;
    const _Float16* p = (const _Float16*)x;
    if (out8 && aligned8(x)) hipLaunchKernelGGL((split_kernel<_Float16, f16x4, true>), g, b, 0, st, p, n, hi, lo);
    else hipLaunchKernelGGL((split_kernel<_Float16, f16x4, false>), g, b, 0, st, p, n, hi, lo);
  } else if (x_dtype == BF16X_F32) {
    if (!aligned4(x)) return BF16X_EARG;
    const float* p = (const float*)x;
    if (out8 && aligned16(x)) hipLaunchKernelGGL((split_kernel<float, f32x4, true>), g, b, 0, st, p, n, hi, lo);
    else hipLaunchKernelGGL((split_kernel<float, f32x4, false>), g, b, 0, st, p, n, hi, lo);
  } else {
    return BF16X_EDTYPE;
  }
  return launch_status();
}

extern "C" int bf16x_add_terms(const float* a, const float* b, int64_t n, void* y, int32_t y_dtype,
                               bf16x_stream_t stream) {
  if (!a || !b || !y || n <= 0) return BF16X_EARG;
  if (!aligned4(a) || !aligned4(b)) return BF16X_EARG;
  hipStream_t st = (hipStream_t)stream;
  const dim3 g(grid_of(n)), bl(256);
  const bool in16 = aligned16(a) && aligned16(b);
  if (y_dtype == BF16X_F16) {
    if (!aligned2(y)) return BF16X_EARG;
    _Float16* p = (_Float16*)y;
    if (in16 && aligned8(y)) hipLaunchKernelGGL((add_kernel<_Float16, f16x4, true>), g, bl, 0, st, a, b, n, p);
    else hipLaunchKernelGGL((add_kernel<_Float16, f16x4, false>), g, bl, 0, st, a, b, n, p);
  } else if (y_dtype == BF16X_F32) {
    if (!aligned4(y)) return BF16X_EARG;
    float* p = (float*)y;
    if (in16 && aligned16(y)) hipLaunchKernelGGL((add_kernel<float, f32x4, true>), g, bl, 0, st, a, b, n, p);
    else hipLaunchKernelGGL((add_kernel<float, f32x4, false>), g, bl, 0, st, a, b, n, p);
  } else {
    return BF16X_EDTYPE;
  }
  return launch_status();
}
