// paged_decode.hip -- single-token paged decode attention with GQA, split-K,
// for gfx950 (CDNA4, wave64).
//
// Pass 1 (decode_stream_kernel, decode_stream.hpp) splits every sequence into
// partitions of P tokens and leaves per (partition, query head) the partial
// softmax state (m, l, acc); sequences that fit one partition are finished
// there.
// Pass 2 (decode_merge_kernel): per (query head, sequence) merge of the
// partition partials m (max), l (sum), acc (unnormalised PV):
//   M = max m_p;  out = sum_p 2^(m_p - M) acc_p / sum_p 2^(m_p - M) l_p.
#include "decode_stream.hpp"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>
#include <type_traits>

namespace rkv {
namespace {

constexpr float kLog2e = 1.4426950408889634f;
// Upper bound on partitions per sequence the merge pass accepts (LDS weights):
// 2.6M tokens at 640 tokens per partition.
constexpr int kMaxMergeParts = 4096;  // 16 KiB of merge weights in LDS

// grid = (num_q_heads, num_seqs), one workgroup of kMergeWaves waves per
// (query head, sequence).  All threads take the partition maxima and the
// weights 2^(m_p - M) (kept in LDS); then lane l of a wave reads float4 c =
// l % (D/4) of partition rows p = l / (D/4) + ..., so one wave instruction
// covers 64 / (D/4) partitions (2 for D = 128) and the kMergeWaves waves
// split the partitions; per-row sums meet through shuffles and LDS.
constexpr int kMergeWaves = 4;

template <int D>
__global__ __launch_bounds__(64 * kMergeWaves) void decode_merge_kernel(
    float* __restrict__ out, const float* __restrict__ part_acc,
    const float* __restrict__ part_ml, const int32_t* __restrict__ ctx_lens, int ctx_cap,
    int num_q_heads, int P, int max_parts) {
  constexpr int NT = 64 * kMergeWaves;
  constexpr int V4 = D / 4;        // float4 per partition row
  constexpr int RPW = 64 / V4;     // partition rows per wave instruction
  extern __shared__ float s_w[];   // max_parts weights (dynamic LDS)
  __shared__ float s_red[kMergeWaves];
  __shared__ __align__(16) float s_acc[kMergeWaves][D];
  const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6;
  int L = ctx_lens[b];
  L = L < 0 ? 0 : (L > ctx_cap ? ctx_cap : L);
  const int np = (L + P - 1) / P;
  if (np <= 1) return;
  const int64_t row0 = ((int64_t)b * num_q_heads + h) * max_parts;
  const int r = lane / V4, c = lane % V4;
  if (np <= kMergeWaves * RPW) {
    // At most one partition row per lane group: the row's acc and its
    // (m, l) are requested together, so the merge waits on memory once.
    __shared__ float s_den[kMergeWaves];
    const int p = w * RPW + r;
    const bool has = p < np;
    const float4 a = has ? *reinterpret_cast<const float4*>(part_acc + (row0 + p) * D + 4 * c)
                         : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float2 ml = has ? *reinterpret_cast<const float2*>(part_ml + (row0 + p) * 2)
                          : make_float2(-INFINITY, 0.0f);
    float M = wave_max(ml.x);
    if (lane == 0) s_red[w] = M;
    __syncthreads();
    M = s_red[0];
#pragma unroll
    for (int x = 1; x < kMergeWaves; ++x) M = fmaxf(M, s_red[x]);
    const float wgt = (ml.x == -INFINITY || M == -INFINITY) ? 0.0f : exp2f(ml.x - M);
    float4 num = make_float4(wgt * a.x, wgt * a.y, wgt * a.z, wgt * a.w);
    const float den = wave_sum(c == 0 ? wgt * ml.y : 0.0f);  // each row's l once
#pragma unroll
    for (int o = V4; o < 64; o <<= 1) {
      num.x += __shfl_xor(num.x, o);
      num.y += __shfl_xor(num.y, o);
      num.z += __shfl_xor(num.z, o);
      num.w += __shfl_xor(num.w, o);
    }
    if (r == 0) *reinterpret_cast<float4*>(&s_acc[w][4 * c]) = num;
    if (lane == 0) s_den[w] = den;
    __syncthreads();
    float dsum = 0.0f;
#pragma unroll
    for (int x = 0; x < kMergeWaves; ++x) dsum += s_den[x];
    for (int dd = tid; dd < D; dd += NT) {
      float v = 0.0f;
#pragma unroll
      for (int x = 0; x < kMergeWaves; ++x) v += s_acc[x][dd];
      out[((int64_t)b * num_q_heads + h) * D + dd] = dsum > 0.0f ? v / dsum : 0.0f;
    }
    return;
  }
  float M = -INFINITY;
  for (int p = tid; p < np; p += NT) M = fmaxf(M, part_ml[(row0 + p) * 2]);
  M = wave_max(M);
  if (lane == 0) s_red[w] = M;
  __syncthreads();
  M = s_red[0];
#pragma unroll
  for (int x = 1; x < kMergeWaves; ++x) M = fmaxf(M, s_red[x]);
  __syncthreads();
  float den = 0.0f;
  for (int p = tid; p < np; p += NT) {
    const float m = part_ml[(row0 + p) * 2];
    const float wgt = (m == -INFINITY || M == -INFINITY) ? 0.0f : exp2f(m - M);
    s_w[p] = wgt;
    den = fmaf(wgt, part_ml[(row0 + p) * 2 + 1], den);
  }
  den = wave_sum(den);
  if (lane == 0) s_red[w] = den;
  __syncthreads();
  den = 0.0f;
#pragma unroll
  for (int x = 0; x < kMergeWaves; ++x) den += s_red[x];
  // weighted sum of the acc rows
  float4 num = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 4
  for (int p = w * RPW + r; p < np; p += kMergeWaves * RPW) {
    const float wgt = s_w[p];
    const float4 a = *reinterpret_cast<const float4*>(part_acc + (row0 + p) * D + 4 * c);
    num.x = fmaf(wgt, a.x, num.x);
    num.y = fmaf(wgt, a.y, num.y);
    num.z = fmaf(wgt, a.z, num.z);
    num.w = fmaf(wgt, a.w, num.w);
  }
#pragma unroll
  for (int o = V4; o < 64; o <<= 1) {
    num.x += __shfl_xor(num.x, o);
    num.y += __shfl_xor(num.y, o);
    num.z += __shfl_xor(num.z, o);
    num.w += __shfl_xor(num.w, o);
  }
  if (r == 0) *reinterpret_cast<float4*>(&s_acc[w][4 * c]) = num;
  __syncthreads();
  for (int dd = tid; dd < D; dd += NT) {
    float v = 0.0f;
#pragma unroll
    for (int x = 0; x < kMergeWaves; ++x) v += s_acc[x][dd];
    out[((int64_t)b * num_q_heads + h) * D + dd] = den > 0.0f ? v / den : 0.0f;
  }
}

// Merge for calls with at most kMergeRowsMaxParts partitions per sequence
// (max_context <= 8 partitions: 64 x U[512, 4096] and most decode batches).  One
// wave per (sequence, query head), four per workgroup, no LDS and no
// barrier: lane l holds float4 c = l % (D/4) of partition rows
// p = l / (D/4) + RPW j, and the rows meet through cross-lane reductions.
// The length and every row the call could have written are requested
// together (rows at or past the sequence's partition count hold stale bytes
// from earlier calls and are removed by selects, never multiplied), so the
// wave waits on memory once.
constexpr int kMergeRowsMaxParts = 8;

// Reduction over the RPW lanes l, l + V4, l + 2 V4, ... (same column c).
template <int V4, bool MAX>
__device__ __forceinline__ float rows_reduce(float x) {
  auto op = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
  if constexpr (V4 <= 8) x = op(x, dpp<0x128>(x));  // lane l ^ 8 inside a 16-lane row
  if constexpr (V4 <= 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

template <int D>
__global__ __launch_bounds__(256) void decode_merge_rows_kernel(
    float* __restrict__ out, const float* __restrict__ part_acc,
    const float* __restrict__ part_ml, const int32_t* __restrict__ ctx_lens, int ctx_cap,
    int num_q_heads, int P, int max_parts, int n_rows) {
  constexpr int V4 = D / 4, RPW = 64 / V4, J = kMergeRowsMaxParts / RPW;
  static_assert(RPW >= 2 && J >= 1, "head_dim 32, 64 or 128");
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);  // sequence * num_q_heads + head
  if (row >= n_rows) return;
  const int b = row / num_q_heads;
  int L = ctx_lens[b];
  const int r = lane / V4, c = lane % V4;
  const int64_t row0 = (int64_t)row * max_parts;
  float4 a[J];
  float2 ml[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int p = r + RPW * j;
    if (p < max_parts) {
      a[j] = *reinterpret_cast<const float4*>(part_acc + (row0 + p) * D + 4 * c);
      ml[j] = *reinterpret_cast<const float2*>(part_ml + (row0 + p) * 2);
    } else {
      a[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      ml[j] = make_float2(-INFINITY, 0.0f);
    }
  }
  L = L < 0 ? 0 : (L > ctx_cap ? ctx_cap : L);
  const int np = (L + P - 1) / P;
  if (np <= 1) return;  // finished by the partition pass
  float m[J], M = -INFINITY;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    m[j] = r + RPW * j < np ? ml[j].x : -INFINITY;
    M = fmaxf(M, m[j]);
  }
  M = rows_reduce<V4, true>(M);
  float4 num = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  float den = 0.0f;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const bool use = m[j] != -INFINITY;  // a written row of a partition with a valid token
    const float w = use ? exp2f(m[j] - M) : 0.0f;
    const float4 x = use ? a[j] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    num.x = fmaf(w, x.x, num.x);
    num.y = fmaf(w, x.y, num.y);
    num.z = fmaf(w, x.z, num.z);
    num.w = fmaf(w, x.w, num.w);
    den = fmaf(w, use ? ml[j].y : 0.0f, den);
  }
  num.x = rows_reduce<V4, false>(num.x);
  num.y = rows_reduce<V4, false>(num.y);
  num.z = rows_reduce<V4, false>(num.z);
  num.w = rows_reduce<V4, false>(num.w);
  den = rows_reduce<V4, false>(den);
  if (r == 0) {
    const float inv = den > 0.0f ? 1.0f / den : 0.0f;
    *reinterpret_cast<float4*>(out + (int64_t)row * D + 4 * c) =
        den > 0.0f ? make_float4(num.x * inv, num.y * inv, num.z * inv, num.w * inv)
                   : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
}

// ---- dispatch ----------------------------------------------------------------

inline bool one_byte(int dtype) { return dtype == RKV_I8 || dtype == RKV_FP8; }

int default_part(int dtype, int /*max_context*/) { return one_byte(dtype) ? kPQ : kP; }

// The partition size rkv_decode_attention uses when the caller leaves it to
// the library: for bf16 pools with head_dim 128 and at most 4 query heads
// per KV head, 1280 when the call holds work for at least 1,200 such
// partitions over all KV heads (contexts taken as uniform up to cap), else
// 768 when it holds work for 1,000 of those, else 640 when it holds work for
// 800 partitions of 512, else 512 (64 x U[512, 4096] 768, 8 x U[16384, 65536]
// and 256 x U[1, 8192] 1280; and, us per call at 512 / 640 /
// 768 over U[512, 4096] contexts, 32 layers back to back: 8 sequences x 8
// KV heads 19.5 / 22.4 / 24.3, 64 x 1 (one GPU's share of 8 KV heads split
// over 8) 23.8 / 24.5 / 25.9, 16 x 8 33.4 / 38.9 / 35.9, 64 x 2 36.9 /
// 41.4 / 40.7, 24 x 8 42.4 / 43.5 / 43.8, 32 x 8 56.4 / 56.5 / 55.7, 64 x 4
// 60.8 / 58.9 / 64.6, 48 x 8 82.8 / 81.7 / 81.3).
// The 512-token tier holds for fp32 pools and every head shape: 512 / 640
// us at 8 and 16 sequences x 8 KV heads, G = 8: 21.9 / 23.7, 32.0 / 37.1;
// head_dim 64: 13.5 / 15.1, 20.6 / 23.6; fp32 pools: 31.8 / 37.3, 58.9 /
// 69.0; at 32 and 64 sequences even or 640 ahead (G = 8 at 64: 121.6 /
// 116.3).
// For 1-byte pools the answer is a size for the caller to ask for (their entry
// points take 640 otherwise): 512 up to twice the work (int8, contexts U[512,
// 4096], 512 / 640: 8 sequences 13.4 / 15.2, 16 sequences 21.0 / 24.2, 32
// sequences 33.0 / 33.8, 64 sequences 66.5 / 64.2; 64 x 1 KV head 16.0 /
// 16.4).  It is no default because it does not hold for every shape: over 404
// shapes of int8 and fp8 it took 0.64 to 1.24 of the time at 640 (median 0.83;
// 128 x U[512, 4096] with one KV head of 64 x 8 queries 21.2 -> 25.4).
// Calls with few workgroups: 512-token partitions leave most CUs idle, so the
// smaller of 128 and 256 tokens is taken that gives at most 256 workgroups (a CU
// each) and at most 128 partitions a sequence.  us per call, partition kernel and
// merge, at 512 tokens / the pick; bf16 pools, head_dim 128, contexts at the cap
// unless given:
//   8 KV heads x 4: 1 sequence of 600 11.5 / 7.6, 4,096 11.8 / 9.6; 2 of U[512,
//   4096] 12.8 / 10.5; 4 of 600 12.3 / 8.7, 1,024 12.0 / 9.2, 2,048 12.6 / 11.6; 8
//   of 600 12.4 / 10.0, 1,024 12.6 / 11.3; 10 of 700 13.0 / 11.3.
//   1 x 4: 1 of 16,384 12.6 / 10.3, 32,768 13.3 / 11.6; 16 of 2,048 12.5 / 10.7,
//   4,096 13.4 / 13.0; 64 of 600 12.9 / 10.8, 1,024 13.0 / 12.3; 85 of 700 13.3 /
//   12.1.  2 x 4: 1 of 32,768 13.9 / 13.7; 32 of 1,024 12.9 / 12.1.  32 x 1: 1 of
//   1,024 10.7 / 8.7, 2 of 1,024 11.5 / 10.6.
// Outside it: 4 of U[512, 4096] 12.7 / 14.2 at 256, 1 of 16,000 16.3 / 17.9; one KV
// head at 65,536 tokens 14.6 / 15.3 at 256 (256 partials to a merge workgroup).
// 0: not such a call.  (One that fits a 512-token partition needs no merge and is
// left alone.)
constexpr int kTinyGroups = 256, kTinyParts = 128;
int tiny_part(int num_seqs, int64_t num_kv_heads, int cap) {
  if (cap <= kSmallP) return 0;
  for (int P = kShortP; P <= 2 * kShortP; P *= 2) {
    const int64_t parts = ((int64_t)cap + P - 1) / P;
    if (parts <= kTinyParts && num_kv_heads * num_seqs * parts <= kTinyGroups) return P;
  }
  return 0;
}

int shape_part(int dtype, int num_seqs, int num_q_heads, int num_kv_heads, int head_dim,
               int cap) {
  if (num_kv_heads <= 0 || num_seqs <= 0 || cap <= 0) return default_part(dtype, cap);
  if (const int tiny = tiny_part(num_seqs, num_kv_heads, cap)) return tiny;
  const double work = (double)num_kv_heads * num_seqs * (0.5 * cap);  // KV-head tokens
  if (work < (one_byte(dtype) ? 1600.0 : 800.0) * kSmallP) return kSmallP;
  if (one_byte(dtype)) return default_part(dtype, cap);
  if (dtype != RKV_BF16 || head_dim != 128 || num_q_heads % num_kv_heads != 0 ||
      num_q_heads / num_kv_heads > 4)
    return default_part(dtype, cap);
  if (work >= 1200.0 * kWideP2) return kWideP2;
  if (work >= 1000.0 * kWideP1) return kWideP1;
  return kP;
}

// The partition size a call uses: the request when it is > 0 (a multiple of
// 16 * SPLIT up to the largest 4-wave build, or for bf16 pools a multiple of
// 128 up to 1280), else the default; a negative status for an unsupported
// request.
int resolve_part(int requested, int dtype, int max_context) {
  if (requested <= 0) return default_part(dtype, max_context);
  const int split = one_byte(dtype) ? RKV_DECODE_SPLIT_Q : RKV_DECODE_SPLIT;
  const int maxp = one_byte(dtype) ? kPQ : kP;
  if (requested % (16 * split) == 0 && requested <= maxp) return requested;
  if (dtype == RKV_BF16 && requested > maxp && requested <= kWideP2 &&
      requested % (16 * kWideSplit) == 0)
    return requested;
  return RKV_ERR_UNSUPPORTED;
}

Launch pick(int dtype, int D, int G, int P, bool append) {
  switch (dtype) {
    case RKV_F32: return decode_f32(D, G, P, append);
    case RKV_BF16: return decode_bf16(D, G, P, append);
    case RKV_I8: return decode_i8(D, G, P, append);
    case RKV_FP8: return decode_fp8(D, G, P, append);
    default: return Launch{};
  }
}

struct DecodeArgs {
  float* out;
  const float* q;
  const void* k_pool;
  const void* v_pool;
  const int32_t* block_tables;
  int max_blocks_per_seq;
  const int32_t* ctx_lens;
  int num_seqs, num_q_heads, num_kv_heads, head_dim, block_size;
  int64_t num_blocks;
  int max_context;
  float scale;
  int dtype, partition_size;
  void* workspace;
  size_t workspace_bytes;
  hipStream_t stream;
  const float* k_scale = nullptr;  // 1-byte pools: [num_blocks][Hkv][block_size] fp32
  const float* v_scale = nullptr;
  const float* k_new = nullptr;  // fused append (bf16 pools): [num_seqs][Hkv][D] fp32
  const float* v_new = nullptr;
};

size_t ws_bytes(int B, int Hq, int D, int max_parts) {
  if (max_parts <= 1) return 0;
  const size_t rows = (size_t)B * Hq * max_parts;
  const size_t acc = rows * D * sizeof(float);
  const size_t acc_pad = (acc + 255) & ~size_t(255);
  return acc_pad + rows * 2 * sizeof(float);
}

// shape_part for a call with this workspace: one sized for 512-token
// partitions (all a call once needed) still takes a call tiny_part would split
// finer, at 512.
int auto_part(int dtype, int num_seqs, int num_q_heads, int num_kv_heads, int head_dim, int cap,
              size_t workspace_bytes) {
  const int P = shape_part(dtype, num_seqs, num_q_heads, num_kv_heads, head_dim, cap);
  if (P < kSmallP && num_q_heads > 0 && head_dim > 0 &&
      ws_bytes(num_seqs, num_q_heads, head_dim, (cap + P - 1) / P) > workspace_bytes)
    return kSmallP;
  return P;
}

int ctx_cap_of(int max_context, int max_blocks_per_seq, int block_size) {
  const int64_t cap = (int64_t)max_blocks_per_seq * block_size;
  return (int)(max_context < cap ? max_context : cap);
}

int validate(const DecodeArgs& a, int& max_parts, int& P) {
  if (a.num_seqs < 0 || a.max_blocks_per_seq < 0 || a.num_blocks < 0)
    return fail(RKV_ERR_INVALID_ARG, "negative size argument");
  if (a.num_q_heads <= 0 || a.num_kv_heads <= 0 || a.num_q_heads % a.num_kv_heads)
    return fail(RKV_ERR_INVALID_ARG, "num_q_heads must be a positive multiple of num_kv_heads");
  const bool q8 = a.dtype == RKV_I8 || a.dtype == RKV_FP8;
  if (a.dtype != RKV_F32 && a.dtype != RKV_BF16 && !q8)
    return fail(RKV_ERR_INVALID_ARG, "dtype must be RKV_F32, RKV_BF16, RKV_I8 or RKV_FP8");
  if (q8 && a.head_dim == 32)
    return fail(RKV_ERR_UNSUPPORTED, "1-byte pools: head_dim must be 64 or 128");
  if (a.block_size != kBS) return fail(RKV_ERR_UNSUPPORTED, "block_size must be 16");
  if (a.head_dim != 32 && a.head_dim != 64 && a.head_dim != 128)
    return fail(RKV_ERR_UNSUPPORTED, "head_dim must be 32, 64 or 128");
  const int G = a.num_q_heads / a.num_kv_heads;
  if (G != 1 && G != 2 && G != 4 && G != 8)
    return fail(RKV_ERR_UNSUPPORTED, "num_q_heads / num_kv_heads must be 1, 2, 4 or 8");
  P = resolve_part(a.partition_size, a.dtype, a.max_context);
  if (P < 0)
    return fail(RKV_ERR_UNSUPPORTED,
                "partition_size must be a multiple of 64 tokens up to 640, for bf16 pools also a "
                "multiple of 128 up to 1280 (or <= 0 for the default)");
  if (a.num_seqs > 65535 || a.num_kv_heads > 65535)
    return fail(RKV_ERR_INVALID_ARG, "num_seqs and num_kv_heads must be <= 65535");
  if (a.max_context < 0) return fail(RKV_ERR_INVALID_ARG, "max_context must be >= 0");
  if (a.num_blocks < 1) return fail(RKV_ERR_INVALID_ARG, "num_blocks must be >= 1");
  const int cap = ctx_cap_of(a.max_context, a.max_blocks_per_seq, a.block_size);
  max_parts = cap <= 0 ? 1 : (cap + P - 1) / P;
  if (max_parts > kMaxMergeParts)
    return fail(RKV_ERR_UNSUPPORTED, "max_context / partition size above 4096 partitions");
  if (a.num_seqs == 0) return RKV_OK;
  if (!a.out || !a.q || !a.k_pool || !a.v_pool || !a.block_tables || !a.ctx_lens)
    return fail(RKV_ERR_INVALID_ARG, "null pointer argument");
  if (q8 && (!a.k_scale || !a.v_scale))
    return fail(RKV_ERR_INVALID_ARG,
                "1-byte pools need their scale pools (rkv_decode_attention_q)");
  if (!aligned16(a.out) || !aligned16(a.q) || !aligned16(a.k_pool) || !aligned16(a.v_pool))
    return fail(RKV_ERR_INVALID_ARG, "out, q and pools must be 16-byte aligned");
  const size_t need = ws_bytes(a.num_seqs, a.num_q_heads, a.head_dim, max_parts);
  if (need > 0 && (!a.workspace || a.workspace_bytes < need))
    return fail(RKV_ERR_WORKSPACE, "workspace missing or smaller than rkv_decode_workspace_bytes()");
  if (need > 0 && !aligned16(a.workspace))
    return fail(RKV_ERR_INVALID_ARG, "workspace must be 16-byte aligned");
  return RKV_OK;
}

void split_ws(void* ws, int B, int Hq, int D, int max_parts, float*& acc, float*& ml) {
  const size_t rows = (size_t)B * Hq * max_parts;
  const size_t acc_pad = (rows * D * sizeof(float) + 255) & ~size_t(255);
  acc = static_cast<float*>(ws);
  ml = reinterpret_cast<float*>(static_cast<char*>(ws) + acc_pad);
}

int launch_partitions(const DecodeArgs& a, int max_parts, int P) {
  const int G = a.num_q_heads / a.num_kv_heads;
  const int cap = ctx_cap_of(a.max_context, a.max_blocks_per_seq, a.block_size);
  // One partition per sequence has to hold the context cap, not P: up to 512
  // tokens the smallest build that does (pick_p).
  if (max_parts == 1 && cap <= kSmallP)
    P = cap <= kShortP ? kShortP : (cap + kShortP - 1) / kShortP * kShortP;
  Launch l = pick(a.dtype, a.head_dim, G, P, a.k_new != nullptr);
  if (!l.kernel) return fail(RKV_ERR_UNSUPPORTED, "no decode kernel for this shape");
  float *acc = nullptr, *ml = nullptr;
  if (max_parts > 1) split_ws(a.workspace, a.num_seqs, a.num_q_heads, a.head_dim, max_parts, acc, ml);
  // KV-head major: the Hkv workgroups of one (partition, sequence) are adjacent
  const dim3 grid((unsigned)a.num_kv_heads, (unsigned)max_parts, (unsigned)a.num_seqs);
  const size_t pad = (a.dtype == RKV_BF16 && a.head_dim == 128) ? RKV_DECODE_LDS_PAD_16 : 0;
  hipLaunchKernelGGL(l.kernel, grid, dim3(l.nw * 64), pad, a.stream, a.out, acc, ml, a.q, a.k_pool,
                     a.v_pool, a.k_scale, a.v_scale, a.block_tables, a.max_blocks_per_seq,
                     a.ctx_lens, cap,
                     a.num_kv_heads, a.num_blocks, a.scale * kLog2e, max_parts,
                     P / (kBS * l.nw), a.k_new, a.v_new);
  return check_launch("decode_stream_kernel");
}

int launch_merge(float* out, const int32_t* ctx_lens, int num_seqs, int num_q_heads, int head_dim,
                 int cap, int P, int max_parts, void* ws, hipStream_t stream) {
  if (max_parts <= 1 || num_seqs == 0) return RKV_OK;
  float *acc = nullptr, *ml = nullptr;
  split_ws(ws, num_seqs, num_q_heads, head_dim, max_parts, acc, ml);
  if (max_parts <= kMergeRowsMaxParts && (int64_t)num_seqs * num_q_heads <= (1 << 28)) {
    const int n_rows = num_seqs * num_q_heads;
    const unsigned nwg = (unsigned)((n_rows + 3) / 4);
    switch (head_dim) {
      case 32:
        decode_merge_rows_kernel<32><<<nwg, 256, 0, stream>>>(out, acc, ml, ctx_lens, cap,
                                                              num_q_heads, P, max_parts, n_rows);
        break;
      case 64:
        decode_merge_rows_kernel<64><<<nwg, 256, 0, stream>>>(out, acc, ml, ctx_lens, cap,
                                                              num_q_heads, P, max_parts, n_rows);
        break;
      default:
        decode_merge_rows_kernel<128><<<nwg, 256, 0, stream>>>(out, acc, ml, ctx_lens, cap,
                                                               num_q_heads, P, max_parts, n_rows);
        break;
    }
    return check_launch("decode_merge_rows_kernel");
  }
  dim3 grid((unsigned)num_q_heads, (unsigned)num_seqs);
  const size_t lds = (size_t)max_parts * sizeof(float);
  switch (head_dim) {
    case 32:
      decode_merge_kernel<32><<<grid, 64 * kMergeWaves, lds, stream>>>(out, acc, ml, ctx_lens, cap, num_q_heads,
                                                       P, max_parts);
      break;
    case 64:
      decode_merge_kernel<64><<<grid, 64 * kMergeWaves, lds, stream>>>(out, acc, ml, ctx_lens, cap, num_q_heads,
                                                       P, max_parts);
      break;
    default:
      decode_merge_kernel<128><<<grid, 64 * kMergeWaves, lds, stream>>>(out, acc, ml, ctx_lens, cap, num_q_heads,
                                                        P, max_parts);
      break;
  }
  return check_launch("decode_merge_kernel");
}

}  // namespace
}  // namespace rkv

using namespace rkv;

extern "C" size_t rkv_decode_workspace_bytes(int num_seqs, int num_q_heads, int head_dim,
                                             int max_context, int partition_size) {
  if (num_seqs <= 0 || num_q_heads <= 0 || head_dim <= 0 || max_context <= 0) return 0;
  // a given partition size, else the most partitions any pick gives a call of up
  // to max_context tokens: the 512-token build's, or tiny_part's at as few KV
  // heads as num_q_heads allows
  const auto parts = [&](int64_t P) { return (max_context + P - 1) / P; };
  if (partition_size > 0)
    return ws_bytes(num_seqs, num_q_heads, head_dim, (int)parts(partition_size));
  const int64_t groups = (int64_t)num_seqs * ((num_q_heads + (int64_t)7) / 8);
  const int64_t tiny =
      max_context <= kSmallP
          ? 1
          : std::min({parts(kShortP), (int64_t)kTinyParts, (int64_t)kTinyGroups / groups});
  static_assert(kSmallP <= kP && kSmallP <= kPQ, "512 tokens is the smallest pick but tiny_part's");
  const int max_parts = (int)std::max(parts(kSmallP), tiny);
  return ws_bytes(num_seqs, num_q_heads, head_dim, max_parts);
}

extern "C" int rkv_decode_partition_size(int partition_size, int head_dim, int dtype,
                                         int max_context) {
  clear_error();
  (void)head_dim;
  if (dtype != RKV_F32 && dtype != RKV_BF16 && !one_byte(dtype))
    return fail(RKV_ERR_INVALID_ARG, "dtype must be RKV_F32, RKV_BF16, RKV_I8 or RKV_FP8");
  const int P = resolve_part(partition_size, dtype, max_context);
  if (P < 0)
    return fail(P, "partition_size must be a multiple of 64 tokens up to 640, for bf16 pools also "
                   "a multiple of 128 up to 1280 (or <= 0)");
  return P;
}

extern "C" int rkv_decode_partition_size_for(int partition_size, int num_seqs, int num_q_heads,
                                             int num_kv_heads, int head_dim, int dtype,
                                             int max_context) {
  clear_error();
  if (dtype != RKV_F32 && dtype != RKV_BF16 && !one_byte(dtype))
    return fail(RKV_ERR_INVALID_ARG, "dtype must be RKV_F32, RKV_BF16, RKV_I8 or RKV_FP8");
  if (partition_size <= 0)
    return shape_part(dtype, num_seqs, num_q_heads, num_kv_heads, head_dim,
                      max_context < 0 ? 0 : max_context);
  const int P = resolve_part(partition_size, dtype, max_context);
  if (P < 0)
    return fail(P, "partition_size must be a multiple of 64 tokens up to 640, for bf16 pools also "
                   "a multiple of 128 up to 1280 (or <= 0)");
  return P;
}

extern "C" int rkv_decode_attention_partitions(
    float* out, const float* q, const void* k_pool, const void* v_pool,
    const int32_t* block_tables, int max_blocks_per_seq, const int32_t* ctx_lens, int num_seqs,
    int num_q_heads, int num_kv_heads, int head_dim, int block_size, int64_t num_blocks,
    int max_context, float scale, int dtype, int partition_size, void* workspace,
    size_t workspace_bytes, void* stream) {
  clear_error();
  DecodeArgs a{out, q, k_pool, v_pool, block_tables, max_blocks_per_seq, ctx_lens, num_seqs,
               num_q_heads, num_kv_heads, head_dim, block_size, num_blocks, max_context, scale,
               dtype, partition_size, workspace, workspace_bytes,
               static_cast<hipStream_t>(stream)};
  int max_parts = 1, P = 0;
  if (int rc = validate(a, max_parts, P)) return rc;
  if (num_seqs == 0) return RKV_OK;
  return launch_partitions(a, max_parts, P);
}

extern "C" int rkv_decode_attention_merge(float* out, const int32_t* ctx_lens,
                                          int max_blocks_per_seq, int num_seqs, int num_q_heads,
                                          int head_dim, int block_size, int max_context,
                                          int dtype, int partition_size, const void* workspace,
                                          size_t workspace_bytes, void* stream) {
  clear_error();
  if (num_seqs < 0 || num_q_heads <= 0 || max_blocks_per_seq < 0 || max_context < 0)
    return fail(RKV_ERR_INVALID_ARG, "bad size argument");
  if (block_size != kBS) return fail(RKV_ERR_UNSUPPORTED, "block_size must be 16");
  if (head_dim != 32 && head_dim != 64 && head_dim != 128)
    return fail(RKV_ERR_UNSUPPORTED, "head_dim must be 32, 64 or 128");
  const int P = resolve_part(partition_size, dtype, max_context);
  if (P < 0)
    return fail(RKV_ERR_UNSUPPORTED,
                "partition_size must be a multiple of 64 tokens up to 640, for bf16 pools also a "
                "multiple of 128 up to 1280 (or <= 0 for the default)");
  if (num_seqs > 65535 || num_q_heads > 65535)
    return fail(RKV_ERR_INVALID_ARG, "num_seqs and num_q_heads must be <= 65535");
  const int cap = ctx_cap_of(max_context, max_blocks_per_seq, block_size);
  const int max_parts = cap <= 0 ? 1 : (cap + P - 1) / P;
  if (max_parts > kMaxMergeParts)
    return fail(RKV_ERR_UNSUPPORTED, "max_context / partition size above 4096 partitions");
  if (max_parts <= 1 || num_seqs == 0) return RKV_OK;
  if (!out || !ctx_lens) return fail(RKV_ERR_INVALID_ARG, "null pointer argument");
  const size_t need = ws_bytes(num_seqs, num_q_heads, head_dim, max_parts);
  if (!workspace || workspace_bytes < need)
    return fail(RKV_ERR_WORKSPACE, "workspace missing or smaller than rkv_decode_workspace_bytes()");
  return launch_merge(out, ctx_lens, num_seqs, num_q_heads, head_dim, cap, P, max_parts,
                      const_cast<void*>(workspace), static_cast<hipStream_t>(stream));
}

extern "C" int rkv_decode_attention(float* out, const float* q, const void* k_pool,
                                    const void* v_pool, const int32_t* block_tables,
                                    int max_blocks_per_seq, const int32_t* ctx_lens, int num_seqs,
                                    int num_q_heads, int num_kv_heads, int head_dim,
                                    int block_size, int64_t num_blocks, int max_context,
                                    float scale, int dtype, int partition_size, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  // both passes take the same explicit partition size: the request, or the
  // size shape_part picks for this call
  const int P =
      partition_size > 0
          ? partition_size
          : auto_part(dtype, num_seqs, num_q_heads, num_kv_heads, head_dim,
                      ctx_cap_of(max_context < 0 ? 0 : max_context,
                                 max_blocks_per_seq < 0 ? 0 : max_blocks_per_seq, block_size),
                      workspace ? workspace_bytes : 0);
  int rc = rkv_decode_attention_partitions(out, q, k_pool, v_pool, block_tables,
                                           max_blocks_per_seq, ctx_lens, num_seqs, num_q_heads,
                                           num_kv_heads, head_dim, block_size, num_blocks,
                                           max_context, scale, dtype, P, workspace,
                                           workspace_bytes, stream);
  if (rc) return rc;
  return rkv_decode_attention_merge(out, ctx_lens, max_blocks_per_seq, num_seqs, num_q_heads,
                                    head_dim, block_size, max_context, dtype, P, workspace,
                                    workspace_bytes, stream);
}

// Decode with the step's K/V append fused in (bf16 pools).  In the partition
// that holds position ctx_lens[b] - 1, the wave whose slice covers it stores
// the rounded new row into the pools from the lanes whose ring loads read
// that row, waits for the stores (vmcnt(0), that wave only), and then
// streams its tiles as usual, reading the new row back with them; so the
// result equals rkv_append of those rows followed by rkv_decode_attention,
// bit for bit, in one launch fewer.
extern "C" int rkv_decode_attention_append(
    float* out, const float* q, void* k_pool, void* v_pool, const float* k_new,
    const float* v_new, const int32_t* block_tables, int max_blocks_per_seq,
    const int32_t* ctx_lens, int num_seqs, int num_q_heads, int num_kv_heads, int head_dim,
    int block_size, int64_t num_blocks, int max_context, float scale, int dtype,
    int partition_size, void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  if (dtype != RKV_BF16)
    return fail(RKV_ERR_UNSUPPORTED,
                "rkv_decode_attention_append: RKV_BF16 pools (1-byte pools: "
                "rkv_decode_attention_append_q)");
  if (num_seqs > 0 && (!k_new || !v_new))
    return fail(RKV_ERR_INVALID_ARG, "null pointer argument");
  if (num_seqs > 0 && (!aligned16(k_new) || !aligned16(v_new)))
    return fail(RKV_ERR_INVALID_ARG, "k_new and v_new must be 16-byte aligned");
  const int P =
      partition_size > 0
          ? partition_size
          : auto_part(dtype, num_seqs, num_q_heads, num_kv_heads, head_dim,
                      ctx_cap_of(max_context < 0 ? 0 : max_context,
                                 max_blocks_per_seq < 0 ? 0 : max_blocks_per_seq, block_size),
                      workspace ? workspace_bytes : 0);
  DecodeArgs a{out, q, k_pool, v_pool, block_tables, max_blocks_per_seq, ctx_lens, num_seqs,
               num_q_heads, num_kv_heads, head_dim, block_size, num_blocks, max_context, scale,
               dtype, P, workspace, workspace_bytes, static_cast<hipStream_t>(stream)};
  a.k_new = k_new;
  a.v_new = v_new;
  int max_parts = 1, P2 = 0;
  if (int rc = validate(a, max_parts, P2)) return rc;
  if (num_seqs == 0) return RKV_OK;
  if (int rc = launch_partitions(a, max_parts, P2)) return rc;
  return launch_merge(out, ctx_lens, num_seqs, num_q_heads, head_dim,
                      ctx_cap_of(max_context, max_blocks_per_seq, block_size), P2, max_parts,
                      workspace, a.stream);
}

// rkv_decode_attention_append for 1-byte pools: the new rows quantized as
// rkv_append_q quantizes them.
extern "C" int rkv_decode_attention_append_q(
    float* out, const float* q, void* k_pool, void* v_pool, float* k_scale, float* v_scale,
    const float* k_new, const float* v_new, const int32_t* block_tables, int max_blocks_per_seq,
    const int32_t* ctx_lens, int num_seqs, int num_q_heads, int num_kv_heads, int head_dim,
    int block_size, int64_t num_blocks, int max_context, float scale, int dtype,
    int partition_size, void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  if (dtype != RKV_I8 && dtype != RKV_FP8)
    return fail(RKV_ERR_INVALID_ARG,
                "rkv_decode_attention_append_q: dtype must be RKV_I8 or RKV_FP8");
  if (num_seqs > 0 && (!k_new || !v_new))
    return fail(RKV_ERR_INVALID_ARG, "null pointer argument");
  if (num_seqs > 0 && (!aligned16(k_new) || !aligned16(v_new)))
    return fail(RKV_ERR_INVALID_ARG, "k_new and v_new must be 16-byte aligned");
  DecodeArgs a{out, q, k_pool, v_pool, block_tables, max_blocks_per_seq, ctx_lens, num_seqs,
               num_q_heads, num_kv_heads, head_dim, block_size, num_blocks, max_context, scale,
               dtype, partition_size, workspace, workspace_bytes,
               static_cast<hipStream_t>(stream), k_scale, v_scale};
  a.k_new = k_new;
  a.v_new = v_new;
  int max_parts = 1, P = 0;
  if (int rc = validate(a, max_parts, P)) return rc;
  if (num_seqs == 0) return RKV_OK;
  if (int rc = launch_partitions(a, max_parts, P)) return rc;
  return launch_merge(out, ctx_lens, num_seqs, num_q_heads, head_dim,
                      ctx_cap_of(max_context, max_blocks_per_seq, block_size), P, max_parts,
                      workspace, a.stream);
}

// ---- the entry point that allocates nothing -----------------------------------
// Callers that cannot allocate device memory (code under HIP graph capture,
// tight serving loops, harnesses that forbid hipMalloc) get the split-K
// partials from a file-scope device array instead of a workspace argument.
// Every GPU the library runs on holds its own copy until the process ends.
// Its address on a device comes from hipGetSymbolAddress (the array's name in
// host code is only a stand-in for the symbol), taken once per device with
// that device current and kept.
constexpr size_t kScratchBytes = size_t(16) << 20;  // 16 MiB
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The scratch array's device address on the device that owns `stream`.
int scratch_for(hipStream_t stream, void** ptr) {
  int dev = -1;
  if (stream) {
    if (hipStreamGetDevice(stream, &dev) != hipSuccess)
      return fail(RKV_ERR_HIP, "rkv_decode_attention_noalloc: hipStreamGetDevice failed");
  } else if (hipGetDevice(&dev) != hipSuccess) {
    return fail(RKV_ERR_HIP, "rkv_decode_attention_noalloc: hipGetDevice failed");
  }
  if (dev < 0 || dev >= kMaxDevices)
    return fail(RKV_ERR_UNSUPPORTED, "rkv_decode_attention_noalloc: device index above 63");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    int cur = -1;
    if (hipGetDevice(&cur) != hipSuccess)
      return fail(RKV_ERR_HIP, "rkv_decode_attention_noalloc: hipGetDevice failed");
    if (cur != dev && hipSetDevice(dev) != hipSuccess)
      return fail(RKV_ERR_HIP, "rkv_decode_attention_noalloc: hipSetDevice failed");
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != dev) (void)hipSetDevice(cur);
    if (e != hipSuccess || !p)
      return fail(RKV_ERR_HIP, std::string("rkv_decode_attention_noalloc: hipGetSymbolAddress: ") +
                                   hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return RKV_OK;
}
}  // namespace

extern "C" size_t rkv_decode_noalloc_max_bytes(void) { return kScratchBytes; }

extern "C" int rkv_decode_attention_noalloc(float* out, const float* q, const void* k_pool,
                                            const void* v_pool, const int32_t* block_tables,
                                            int max_blocks_per_seq, const int32_t* ctx_lens,
                                            int num_seqs, int num_q_heads, int num_kv_heads,
                                            int head_dim, int block_size, int64_t num_blocks,
                                            int max_context, float scale, int dtype,
                                            int partition_size, void* stream) {
  clear_error();
  const int cap = ctx_cap_of(max_context < 0 ? 0 : max_context, max_blocks_per_seq < 0 ? 0 : max_blocks_per_seq,
                             block_size);
  // the size rkv_decode_attention will use (the request, or its shape's pick)
  const int P = partition_size > 0
                    ? resolve_part(partition_size, dtype, max_context)
                    : shape_part(dtype, num_seqs, num_q_heads, num_kv_heads, head_dim, cap);
  if (P < 0)
    return fail(RKV_ERR_UNSUPPORTED,
                "partition_size must be a multiple of 64 tokens up to 640, for bf16 pools also a "
                "multiple of 128 up to 1280 (or <= 0 for the default)");
  const int max_parts = cap <= 0 ? 1 : (cap + P - 1) / P;
  const size_t need = (num_seqs > 0 && num_q_heads > 0 && head_dim > 0)
                          ? ws_bytes(num_seqs, num_q_heads, head_dim, max_parts)
                          : 0;
  if (need > kScratchBytes)
    return fail(RKV_ERR_WORKSPACE,
                "rkv_decode_attention_noalloc: split-K partials need " + std::to_string(need) +
                    " bytes, above the 16 MiB scratch (use rkv_decode_attention with a workspace)");
  void* ws = nullptr;
  if (need > 0)
    if (int rc = scratch_for(static_cast<hipStream_t>(stream), &ws)) return rc;
  return rkv_decode_attention(out, q, k_pool, v_pool, block_tables, max_blocks_per_seq, ctx_lens,
                              num_seqs, num_q_heads, num_kv_heads, head_dim, block_size,
                              num_blocks, max_context, scale, dtype, P, ws,
                              need > 0 ? kScratchBytes : 0, stream);
}

extern "C" int rkv_decode_attention_q(float* out, const float* q, const void* k_pool,
                                      const void* v_pool, const float* k_scale,
                                      const float* v_scale, const int32_t* block_tables,
                                      int max_blocks_per_seq, const int32_t* ctx_lens,
                                      int num_seqs, int num_q_heads, int num_kv_heads,
                                      int head_dim, int block_size, int64_t num_blocks,
                                      int max_context, float scale, int dtype,
                                      int partition_size, void* workspace,
                                      size_t workspace_bytes, void* stream) {
  clear_error();
  if (dtype != RKV_I8 && dtype != RKV_FP8)
    return fail(RKV_ERR_INVALID_ARG, "rkv_decode_attention_q: dtype must be RKV_I8 or RKV_FP8");
  DecodeArgs a{out, q, k_pool, v_pool, block_tables, max_blocks_per_seq, ctx_lens, num_seqs,
               num_q_heads, num_kv_heads, head_dim, block_size, num_blocks, max_context, scale,
               dtype, partition_size, workspace, workspace_bytes,
               static_cast<hipStream_t>(stream), k_scale, v_scale};
  int max_parts = 1, P = 0;
  if (int rc = validate(a, max_parts, P)) return rc;
  if (num_seqs == 0) return RKV_OK;
  if (int rc = launch_partitions(a, max_parts, P)) return rc;
  const int cap = ctx_cap_of(max_context, max_blocks_per_seq, block_size);
  return launch_merge(out, ctx_lens, num_seqs, num_q_heads, head_dim, cap, P, max_parts,
                      workspace, a.stream);
}
