// model_ops.hpp -- what projection.hip, model_ops.hip, the decoder and the serving
// engine share.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace rkv {

// rkv_linear with a fused epilogue: epi 0 y = x W^T + b; 1 y = res + (x W^T + b)
// (residual add, y may alias res); 2 y = gelu(x W^T + b).  With ln_g / ln_b
// the input rows are layer-normed first (eps).  The same arithmetic, in the
// same order, as rkv_layer_norm, rkv_linear and then rkv_add / rkv_gelu.
int linear_launch(float* y, const float* x, const float* w, const float* b, const float* res,
                  int epi, int rows, int in_dim, int out_dim, hipStream_t s,
                  const float* ln_g = nullptr, const float* ln_b = nullptr, float eps = 0.0f);

// rkv_argmax of one row of logits and rkv_embed of the winner (pe_row: its
// position's row of the positional table) in one launch.
int argmax_embed_launch(int32_t* id, float* x_next, const float* logits, int vocab,
                        const float* table, const float* pe_row, int dim, hipStream_t s);

// 0.5 v (1 + tanh(sqrt(2 / pi) (v + 0.044715 v^3))), the reference's order.
__device__ __forceinline__ float gelu_f(float v) {
#pragma clang fp contract(off)
  const float k = sqrtf(2.0f / 3.14159265358979323846f);
  const float x3 = v * v * v;
  const float xp = v + 0.044715f * x3;
  const float t = tanhf(k * xp);
  return 0.5f * v * (1.0f + t);
}

// Calls f(std::integral_constant<int, I>) for I = B .. E-1 in order.
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

}  // namespace rkv
