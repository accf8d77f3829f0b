// model_ops.hip -- the fp32 TensorOps subset a decoder step needs on gfx950
// (include/rustral_model.h): embedding + positional term, layer norm, gelu,
// add, argmax, and the per-head attention recipe's matmul, transpose,
// mul_scalar and softmax_dim (projection.hip has linear and its fused forms).
//
// These are not the hot path (the KV cache and decode attention are); they
// exist so a whole decoder step runs on the device.  Each op keeps the
// reference's summation order: one thread owns one output and adds its terms
// serially, with floating-point contraction off, so the results are the bits
// the ndarray backend computes (except gelu's tanh, from the device library).
#include "model_ops.hpp"

#include <cmath>
#include <type_traits>

namespace rkv {
namespace {

__global__ __launch_bounds__(256) void embed_kernel(float* __restrict__ out,
                                                    const float* __restrict__ table,
                                                    const int32_t* __restrict__ ids,
                                                    const float* __restrict__ pe,
                                                    const int32_t* __restrict__ positions,
                                                    int n_tokens, int vocab, int dim,
                                                    int max_len) {
#pragma clang fp contract(off)
  const int t = blockIdx.y;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_tokens || i >= dim) return;
  const int id = ids[t];
  float v = NAN;
  if (id >= 0 && id < vocab) {
    v = table[(int64_t)id * dim + i];
    if (pe) {
      const int p = positions[t];
      v = (p >= 0 && p < max_len) ? v + pe[(int64_t)p * dim + i] : NAN;
    }
  }
  out[(int64_t)t * dim + i] = v;
}

// One wave per row: the row is staged in LDS, lane 0 forms the serial sums
// from it, every lane writes outputs.
__global__ __launch_bounds__(64) void layer_norm_kernel(float* __restrict__ y,
                                                        const float* __restrict__ x,
                                                        const float* __restrict__ g,
                                                        const float* __restrict__ b, int rows,
                                                        int dim, float eps) {
#pragma clang fp contract(off)
  __shared__ float s_stat[2];
  __shared__ float s_row[8192];
  const int r = blockIdx.x, lane = threadIdx.x;
  if (r >= rows) return;
  const float* xr = x + (int64_t)r * dim;
  for (int i = lane; i < dim; i += 64) s_row[i] = xr[i];
  __syncthreads();
  if (lane == 0) {
    float sum = 0.0f;
    for (int i = 0; i < dim; ++i) sum += s_row[i];
    const float mean = sum / (float)dim;
    float vs = 0.0f;
    for (int i = 0; i < dim; ++i) {
      const float t = s_row[i] - mean;
      vs += t * t;
    }
    s_stat[0] = mean;
    s_stat[1] = sqrtf(vs / (float)dim + eps);
  }
  __syncthreads();
  const float mean = s_stat[0], sd = s_stat[1];
  for (int i = lane; i < dim; i += 64) y[(int64_t)r * dim + i] = (s_row[i] - mean) / sd * g[i] + b[i];
}

__global__ __launch_bounds__(256) void gelu_kernel(float* __restrict__ y,
                                                   const float* __restrict__ x, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  y[i] = gelu_f(x[i]);
}

// y may alias a or b (in-place residual add)
__global__ __launch_bounds__(256) void add_kernel(float* y, const float* a, const float* b,
                                                  int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = a[i] + b[i];
}

__global__ __launch_bounds__(256) void mul_scalar_kernel(float* y, const float* x, float s,
                                                         int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = x[i] * s;
}

// Softmax along an axis of `axis` elements at stride `inner` (CpuOps::
// softmax_dim's loops): max over the line with NaN skipped (f32::max /
// fmaxf), e = exp(x - max) written out and added serially in axis order,
// then every e scaled by 1 / sum.
//
// Strided lines (inner > 1): one thread per line, lanes on consecutive i, so
// every step of the three serial loops is a coalesced row access.
__global__ __launch_bounds__(256) void softmax_strided_kernel(float* y, const float* x,
                                                              int64_t lines, int64_t axis,
                                                              int64_t inner) {
#pragma clang fp contract(off)
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= lines) return;
  const int64_t o = g / inner, i = g - o * inner;
  const float* xl = x + o * axis * inner + i;
  float* yl = y + o * axis * inner + i;
  float mx = -INFINITY;
  for (int64_t a = 0; a < axis; ++a) mx = fmaxf(mx, xl[a * inner]);
  float sum = 0.0f;
  for (int64_t a = 0; a < axis; ++a) {
    const float e = expf(xl[a * inner] - mx);
    yl[a * inner] = e;
    sum += e;
  }
  const float inv = 1.0f / sum;
  for (int64_t a = 0; a < axis; ++a) yl[a * inner] *= inv;
}

// Contiguous lines (inner == 1): one 256-thread workgroup per row.  The max
// is a tree over the workgroup (max is exact, so any order gives the serial
// scan's value); the exps are computed in parallel, kChunk at a time, into
// LDS and y, and lane 0 adds each chunk in index order, so the sum is the
// reference's serial sum.  Each thread scales the entries it wrote itself.
constexpr int kSoftmaxChunk = 2048;

__global__ __launch_bounds__(256) void softmax_rows_kernel(float* y, const float* x,
                                                           int64_t axis) {
#pragma clang fp contract(off)
  __shared__ float s_e[kSoftmaxChunk];
  __shared__ float s_red[4];
  __shared__ float s_sum;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const float* xr = x + (int64_t)blockIdx.x * axis;
  float* yr = y + (int64_t)blockIdx.x * axis;
  float mx = -INFINITY;
  for (int64_t a = t; a < axis; a += 256) mx = fmaxf(mx, xr[a]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  if (lane == 0) s_red[w] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
  float sum = 0.0f;  // lane 0 of wave 0 only
  for (int64_t c0 = 0; c0 < axis; c0 += kSoftmaxChunk) {
    const int n = (int)((axis - c0) < kSoftmaxChunk ? (axis - c0) : kSoftmaxChunk);
    for (int j = t; j < n; j += 256) {
      const float e = expf(xr[c0 + j] - mx);
      s_e[j] = e;
      yr[c0 + j] = e;
    }
    __syncthreads();
    if (t == 0)
      for (int j = 0; j < n; ++j) sum += s_e[j];
    __syncthreads();
  }
  if (t == 0) s_sum = sum;
  __syncthreads();
  const float inv = 1.0f / s_sum;
  for (int64_t c0 = 0; c0 < axis; c0 += kSoftmaxChunk) {
    const int n = (int)((axis - c0) < kSoftmaxChunk ? (axis - c0) : kSoftmaxChunk);
    for (int j = t; j < n; j += 256) yr[c0 + j] *= inv;
  }
}

// y[m][n] = sum_k a[m][k] * b[k][n], the sum serial in k (the reference's
// naive loop order) and without contraction.  16 x 16 outputs per workgroup,
// one per thread; k advances through 16-wide tiles of a and b staged in LDS.
constexpr int kMmTile = 16;

__global__ __launch_bounds__(256) void matmul_kernel(float* __restrict__ y,
                                                     const float* __restrict__ a,
                                                     const float* __restrict__ b, int m, int k,
                                                     int n) {
#pragma clang fp contract(off)
  __shared__ float s_a[kMmTile][kMmTile + 1];
  __shared__ float s_b[kMmTile][kMmTile + 1];
  const int tx = threadIdx.x & (kMmTile - 1), ty = threadIdx.x / kMmTile;
  const int row = blockIdx.y * kMmTile + ty, col = blockIdx.x * kMmTile + tx;
  float sum = 0.0f;
  for (int k0 = 0; k0 < k; k0 += kMmTile) {
    s_a[ty][tx] = (row < m && k0 + tx < k) ? a[(int64_t)row * k + k0 + tx] : 0.0f;
    s_b[ty][tx] = (k0 + ty < k && col < n) ? b[(int64_t)(k0 + ty) * n + col] : 0.0f;
    __syncthreads();
    const int kt = (k - k0) < kMmTile ? (k - k0) : kMmTile;
    for (int j = 0; j < kt; ++j) sum += s_a[ty][j] * s_b[j][tx];
    __syncthreads();
  }
  if (row < m && col < n) y[(int64_t)row * n + col] = sum;
}

// y[n][m] = x[m][n]: 32 x 32 tiles through LDS (one padding column keeps the
// transposed reads off a single bank), both sides coalesced.
__global__ __launch_bounds__(256) void transpose_kernel(float* __restrict__ y,
                                                        const float* __restrict__ x, int m,
                                                        int n) {
  __shared__ float s_t[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8 threads
  const int r0 = blockIdx.y * 32, c0 = blockIdx.x * 32;
  for (int r = ty; r < 32; r += 8)
    if (r0 + r < m && c0 + tx < n) s_t[r][tx] = x[(int64_t)(r0 + r) * n + c0 + tx];
  __syncthreads();
  for (int c = ty; c < 32; c += 8)
    if (c0 + c < n && r0 + tx < m) y[(int64_t)(c0 + c) * m + r0 + tx] = s_t[tx][c];
}

// NW waves per row.  Without NaN: each thread scans its elements (i = t,
// t + 64 NW, ...) keeping the last maximum, then lanes and waves combine (larger
// value, or the larger index on a tie).  With a NaN anywhere the answer depends
// on the scan order, so thread 0 repeats the reference's left-to-right scan.
// EMBED: the row's winner is a token id and its embedding row (plus the
// positional one) follows in the same launch, as rkv_embed writes it.
struct EmbedTail {
  float* x;            // [dim]
  const float* table;  // [vocab][dim]
  const float* pe;     // the position's row
  int dim;
};

template <int NW, bool EMBED>
__global__ __launch_bounds__(64 * NW) void argmax_kernel(int32_t* __restrict__ out,
                                                         const float* __restrict__ x, int n,
                                                         EmbedTail tail) {
#pragma clang fp contract(off)
  __shared__ float s_v[NW];
  __shared__ int s_i[NW], s_nan[NW], s_best;
  const int r = blockIdx.x, t = threadIdx.x, lane = t & 63, w = t >> 6;
  const float* xr = x + (int64_t)r * n;
  bool nan = false;
  float bv = -INFINITY;
  int bi = -1;
#pragma unroll 4
  for (int i = t; i < n; i += 64 * NW) {
    const float v = xr[i];
    nan |= v != v;
    if (bi < 0 || v >= bv) {
      bv = v;
      bi = i;
    }
  }
  auto merge = [&](float ov, int oi) {
    if (oi >= 0 && (bi < 0 || ov > bv || (ov == bv && oi > bi))) {
      bv = ov;
      bi = oi;
    }
  };
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float ov = __shfl_xor(bv, o);
    merge(ov, __shfl_xor(bi, o));
  }
  bool any = __ballot(nan) != 0;
  if constexpr (NW > 1) {
    if (lane == 0) {
      s_v[w] = bv;
      s_i[w] = bi;
      s_nan[w] = any;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NW; ++k) any |= s_nan[k] != 0;
  }
  if (t == 0) {
    int best;
    if (any) {
      best = 0;
      for (int i = 1; i < n; ++i)
        if (!(xr[best] > xr[i])) best = i;
    } else {
#pragma unroll
      for (int k = 1; k < NW; ++k) merge(s_v[k], s_i[k]);
      best = bi;
    }
    out[r] = best;
    if constexpr (EMBED) s_best = best;
  }
  if constexpr (EMBED) {
    __syncthreads();
    const float* row = tail.table + (int64_t)s_best * tail.dim;
    for (int i = t; i < tail.dim; i += 64 * NW) tail.x[i] = row[i] + tail.pe[i];
  }
}

unsigned blocks_for(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

int argmax_embed_launch(int32_t* id, float* x_next, const float* logits, int vocab,
                        const float* table, const float* pe_row, int dim, hipStream_t s) {
  argmax_kernel<4, true><<<1, 256, 0, s>>>(id, logits, vocab, EmbedTail{x_next, table, pe_row, dim});
  return check_launch("argmax_embed");
}

}  // namespace rkv

using namespace rkv;

extern "C" int rkv_embed(float* out, const float* table, const int32_t* ids, const float* pe,
                         const int32_t* positions, int n_tokens, int vocab, int dim, int max_len,
                         void* stream) {
  clear_error();
  if (n_tokens < 0 || vocab <= 0 || dim <= 0 || (pe && max_len <= 0))
    return fail(RKV_ERR_INVALID_ARG, "rkv_embed: bad size argument");
  if (n_tokens == 0) return RKV_OK;
  if (n_tokens > 65535) return fail(RKV_ERR_INVALID_ARG, "rkv_embed: n_tokens must be <= 65535");
  if (!out || !table || !ids || (pe && !positions))
    return fail(RKV_ERR_INVALID_ARG, "rkv_embed: null pointer argument");
  embed_kernel<<<dim3(blocks_for(dim, 256), (unsigned)n_tokens), 256, 0,
                 static_cast<hipStream_t>(stream)>>>(out, table, ids, pe, positions, n_tokens,
                                                     vocab, dim, max_len);
  return check_launch("rkv_embed");
}

extern "C" int rkv_layer_norm(float* y, const float* x, const float* g, const float* b, int rows,
                              int dim, float eps, void* stream) {
  clear_error();
  if (rows < 0 || dim <= 0 || dim > 8192)
    return fail(RKV_ERR_INVALID_ARG, "rkv_layer_norm: bad size argument");
  if (rows == 0) return RKV_OK;
  if (!y || !x || !g || !b) return fail(RKV_ERR_INVALID_ARG, "rkv_layer_norm: null pointer");
  layer_norm_kernel<<<(unsigned)rows, 64, 0, static_cast<hipStream_t>(stream)>>>(y, x, g, b, rows,
                                                                               dim, eps);
  return check_launch("rkv_layer_norm");
}

extern "C" int rkv_gelu(float* y, const float* x, int64_t n, void* stream) {
  clear_error();
  if (n < 0) return fail(RKV_ERR_INVALID_ARG, "rkv_gelu: n < 0");
  if (n == 0) return RKV_OK;
  if (!y || !x) return fail(RKV_ERR_INVALID_ARG, "rkv_gelu: null pointer argument");
  gelu_kernel<<<blocks_for(n, 256), 256, 0, static_cast<hipStream_t>(stream)>>>(y, x, n);
  return check_launch("rkv_gelu");
}

extern "C" int rkv_add(float* y, const float* a, const float* b, int64_t n, void* stream) {
  clear_error();
  if (n < 0) return fail(RKV_ERR_INVALID_ARG, "rkv_add: n < 0");
  if (n == 0) return RKV_OK;
  if (!y || !a || !b) return fail(RKV_ERR_INVALID_ARG, "rkv_add: null pointer argument");
  add_kernel<<<blocks_for(n, 256), 256, 0, static_cast<hipStream_t>(stream)>>>(y, a, b, n);
  return check_launch("rkv_add");
}

extern "C" int rkv_mul_scalar(float* y, const float* x, float s, int64_t n, void* stream) {
  clear_error();
  if (n < 0) return fail(RKV_ERR_INVALID_ARG, "rkv_mul_scalar: n < 0");
  if (n == 0) return RKV_OK;
  if (!y || !x) return fail(RKV_ERR_INVALID_ARG, "rkv_mul_scalar: null pointer argument");
  if (n > (int64_t)INT32_MAX * 256) return fail(RKV_ERR_INVALID_ARG, "rkv_mul_scalar: n too large");
  mul_scalar_kernel<<<blocks_for(n, 256), 256, 0, static_cast<hipStream_t>(stream)>>>(y, x, s, n);
  return check_launch("rkv_mul_scalar");
}

extern "C" int rkv_softmax_dim(float* y, const float* x, int64_t outer, int64_t axis,
                               int64_t inner, void* stream) {
  clear_error();
  if (outer < 0 || inner < 0 || axis <= 0)
    return fail(RKV_ERR_INVALID_ARG, "rkv_softmax_dim: bad size argument (axis size must be > 0)");
  if (outer == 0 || inner == 0) return RKV_OK;
  if (!y || !x) return fail(RKV_ERR_INVALID_ARG, "rkv_softmax_dim: null pointer argument");
  if (outer > INT64_MAX / axis || outer * axis > INT64_MAX / inner)
    return fail(RKV_ERR_INVALID_ARG, "rkv_softmax_dim: element count overflows int64");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (inner == 1) {
    if (outer > INT32_MAX) return fail(RKV_ERR_INVALID_ARG, "rkv_softmax_dim: too many rows");
    softmax_rows_kernel<<<(unsigned)outer, 256, 0, s>>>(y, x, axis);
  } else {
    const int64_t lines = outer * inner;
    if (lines > (int64_t)INT32_MAX * 256)
      return fail(RKV_ERR_INVALID_ARG, "rkv_softmax_dim: too many lines");
    softmax_strided_kernel<<<blocks_for(lines, 256), 256, 0, s>>>(y, x, lines, axis, inner);
  }
  return check_launch("rkv_softmax_dim");
}

extern "C" int rkv_matmul(float* y, const float* a, const float* b, int m, int k, int n,
                          void* stream) {
  clear_error();
  if (m < 0 || k < 0 || n < 0) return fail(RKV_ERR_INVALID_ARG, "rkv_matmul: bad size argument");
  if (m == 0 || n == 0) return RKV_OK;
  if (!y || (k > 0 && (!a || !b)))
    return fail(RKV_ERR_INVALID_ARG, "rkv_matmul: null pointer argument");
  if ((m + kMmTile - 1) / kMmTile > 65535)
    return fail(RKV_ERR_INVALID_ARG, "rkv_matmul: m must be <= 1048560");
  const dim3 grid(blocks_for(n, kMmTile), (unsigned)((m + kMmTile - 1) / kMmTile));
  matmul_kernel<<<grid, 256, 0, static_cast<hipStream_t>(stream)>>>(y, a, b, m, k, n);
  return check_launch("rkv_matmul");
}

extern "C" int rkv_transpose(float* y, const float* x, int m, int n, void* stream) {
  clear_error();
  if (m < 0 || n < 0) return fail(RKV_ERR_INVALID_ARG, "rkv_transpose: bad size argument");
  if (m == 0 || n == 0) return RKV_OK;
  if (!y || !x) return fail(RKV_ERR_INVALID_ARG, "rkv_transpose: null pointer argument");
  if (y == x) return fail(RKV_ERR_INVALID_ARG, "rkv_transpose: y must not alias x");
  if ((m + 31) / 32 > 65535) return fail(RKV_ERR_INVALID_ARG, "rkv_transpose: m must be <= 2097120");
  const dim3 grid(blocks_for(n, 32), (unsigned)((m + 31) / 32));
  transpose_kernel<<<grid, 256, 0, static_cast<hipStream_t>(stream)>>>(y, x, m, n);
  return check_launch("rkv_transpose");
}

extern "C" int rkv_argmax(int32_t* out, const float* x, int rows, int n, void* stream) {
  clear_error();
  if (rows < 0 || n <= 0) return fail(RKV_ERR_INVALID_ARG, "rkv_argmax: bad size argument");
  if (rows == 0) return RKV_OK;
  if (!out || !x) return fail(RKV_ERR_INVALID_ARG, "rkv_argmax: null pointer argument");
  const hipStream_t s = static_cast<hipStream_t>(stream);
  // Four waves cut a long row's chain of loads (us, four / one: 1 row of 2,000
  // 3.9 / 4.4, of 32,000 9.4 / 25.6); up to 1,024 columns they only cost
  // workgroups (1 x 1,000 3.6 / 3.7; 4,096 x 256 6.7 / 4.3; 65,536 x 100 51 /
  // 19), and up to 2,048 where the rows fill the chip (2,048 x 2,000 5.8 / 7.2,
  // 4,096 x 2,000 10.1 / 8.4, 65,536 x 2,000 139 / 98; 4,096 columns alike or
  // ahead with four).  2^24 rows of four waves would be 2^32 threads, at which a
  // grid wraps.
  if (n <= 1024 || (n <= 2048 && rows >= 4096) || rows >= 1 << 24)
    argmax_kernel<1, false><<<(unsigned)rows, 64, 0, s>>>(out, x, n, EmbedTail{});
  else
    argmax_kernel<4, false><<<(unsigned)rows, 256, 0, s>>>(out, x, n, EmbedTail{});
  return check_launch("rkv_argmax");
}
