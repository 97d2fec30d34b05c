// conv_mfma.h -- square-kernel convolutions over large planes: ungrouped ones on the matrix cores,
// depthwise ones in tiles (internal to the library; conv.hip chooses).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.h"

namespace oxh {
namespace conv_mfma {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// acc += a x b (v_mfma_f32_32x32x2_f32) in the lanes, columns of the result, that are `in`; the
// others keep acc.
__device__ __forceinline__ void multiply_in(float a, float b, bool in, f32x16 &acc) {
  const f32x16 next = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = in ? next[r] : acc[r];
}

// One group, kernel k x k, the shape checks of conv.hip passed.
struct Dims {
  uint32_t batch, in_c, h, w, out_c, k, stride, pad, oh, ow;
};

// Whether the forward / input gradient of this convolution runs here (K x K: kernel 3 or 5, or
// a strided or padded 1 x 1).
bool takes_forward(const Dims &d);
bool takes_input_backward(const Dims &d);

// y[n][oc][p] = bias[oc] + sum over (ic, tap) of x * weight.
void forward(hipStream_t s, const Dims &d, const float *x, const float *weight,
             const float *bias, float *y);
// dx[n][ic][p] = sum over (oc, tap) of gradient * weight (+ addend, which may be dx itself).
void input_backward(hipStream_t s, const Dims &d, const float *gradient, const float *weight,
                    const float *addend, float *dx);

// A 1 x 1 convolution as a product: y[n][m][p] = bias[m] + sum over k of w[m][k] x[n][k][p] +
// addend (bias and addend may be null, addend may be y), with w[m][k] at weight[m * k_count + k]
// or, transposed (an input gradient: k the output channels), weight[k * m_count + m].
bool takes_pointwise(uint64_t images, uint64_t plane, uint64_t k, uint64_t m);
void pointwise(hipStream_t s, uint32_t images, uint32_t plane, uint32_t k, uint32_t m,
               bool transposed, const float *x, const float *weight, const float *bias,
               const float *addend, float *y);

// Weight gradient of an ungrouped convolution with any kernel.
struct WeightDims {
  uint32_t batch, in_c, h, w, out_c, kh, kw, stride, pad, oh, ow;
};
// Partial sums it leaves, each of out_c * in_c * kh * kw values (1: the gradient itself); 0 when
// the shape does not run here.
uint32_t weight_partials(const WeightDims &d);
// An estimate of its time in us, for a shape that runs here: the layout's cycles at 2.4 GHz, 1.8
// times which, and 5 us, is what 1050 random layers took (within 1.4 times in nine of ten).
double weight_time(const WeightDims &d);
void weight_backward(hipStream_t s, const WeightDims &d, const float *gradient, const float *x,
                     float *out);

// Depthwise convolutions (in_c == out_c == groups) with kernel 3 or 5 and stride 1 or 2
// (conv_depthwise.hip).  addend as in input_backward.
bool takes_depthwise(const Dims &d);
void depthwise_forward(hipStream_t s, const Dims &d, const float *x, const float *weight,
                       const float *bias, float *y);
void depthwise_input_backward(hipStream_t s, const Dims &d, const float *gradient,
                              const float *weight, const float *addend, float *dx);
// Partial sums the weight gradient leaves, each of in_c * k * k values (1: the gradient itself).
uint32_t depthwise_weight_partials(const Dims &d);
void depthwise_weight_backward(hipStream_t s, const Dims &d, const float *gradient,
                               const float *x, float *out);

}  // namespace conv_mfma
}  // namespace oxh
