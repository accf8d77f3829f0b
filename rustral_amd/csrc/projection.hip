// projection.hip -- y = x W^T + b and its fused forms (layer norm before;
// residual add, GELU or the q / k / v split with the KV append after) for
// gfx950, with the reference's serial-order fp32 sums.
//
// Every output is one sum over the input features in index order, each term
// rounded as a product and then added (no fused multiply-add): the bits of the
// reference's CPU loops.  So a sum cannot be split, and a term costs a
// multiplication and an addition, and a wave issues one vector instruction
// per 4 cycles: of a wave of one row's 15 cycles a term (SQ counters, n = 4,096)
// it issues in 9.  With four rows per wave the multiplications run on the
// matrix cores instead:
// v_mfma_f32_4x4x1_16b_f32 with C = 0 gives 256 products fma(x, w, 0), each
// rounded once (checked bit for bit on gfx950, denormals included; the sign
// of a zero product may differ, which no sum that starts at +0 shows), and
// the vector unit only adds: 37 cycles a term for the four rows, 21 of them
// issuing.
#include <cmath>

#include "model_ops.hpp"

namespace rkv {
namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

// What follows the sum.
enum Mode {
  kPlain,     // y = sum + b
  kResidual,  // y = res + (sum + b); y may be res
  kGelu,      // y = gelu(sum + b)
  kQkvF32,    // the q / k / v columns of a layer: q to y, k and v to the
  kQkvBf16,   // token's rows of the pools
};

struct ProjArgs {
  float* y;
  const float* x;
  const float* w;  // [cols][n]; kQkv: wq
  const float* b;
  const float* res;
  const float *ln_g, *ln_b;
  float eps;
  int mode, rows, n, cols;
  // kQkv
  const float *wk, *bk, *wv, *bv;
  void *k_pool, *v_pool;
  const int64_t* slots;
  int q_dim, kvd, num_kv_heads, head_dim, block_size;
  int hd_log2, bs_log2;  // of powers of two, else -1
  int64_t num_slots;
};

// Weight row of output column o.
__device__ __forceinline__ const float* weight_row(const ProjArgs& a, int o) {
  const float* w = a.w;
  if (a.mode >= kQkvF32 && o >= a.q_dim) {
    o -= a.q_dim;
    w = o < a.kvd ? a.wk : a.wv;
    if (o >= a.kvd) o -= a.kvd;
  }
  return w + (int64_t)o * a.n;
}

// What put needs of column o and row r besides the sum, read before the sums
// start so that the end of a wave does not wait for memory again.
struct ColTail {
  float b;     // bias (0 with has_b false)
  bool has_b;
};
struct RowTail {
  float res;     // kResidual
  int64_t slot;  // kQkv
};
__device__ __forceinline__ ColTail col_tail(const ProjArgs& a, int o) {
  const float* b = a.b;
  if (a.mode >= kQkvF32 && o >= a.q_dim) {
    o -= a.q_dim;
    b = o < a.kvd ? a.bk : a.bv;
    if (o >= a.kvd) o -= a.kvd;
  }
  return ColTail{b ? b[o] : 0.0f, b != nullptr};
}
__device__ __forceinline__ RowTail row_tail(const ProjArgs& a, int r, int o) {
  return RowTail{a.mode == kResidual ? a.res[(int64_t)r * a.cols + o] : 0.0f,
                 a.mode >= kQkvF32 ? a.slots[r] : 0};
}

__device__ __forceinline__ void put(const ProjArgs& a, int r, int o, float sum, const ColTail& c,
                                    const RowTail& t) {
#pragma clang fp contract(off)
  const float v = c.has_b ? sum + c.b : sum;
  if (a.mode >= kQkvF32) {
    if (o < a.q_dim) {
      a.y[(int64_t)r * a.q_dim + o] = v;
      return;
    }
    const bool is_v = o >= a.q_dim + a.kvd;
    const int col = o - a.q_dim - (is_v ? a.kvd : 0);
    const int64_t slot = t.slot;
    if (slot < 0 || slot >= a.num_slots) return;  // padding or out-of-range slot
    const int64_t blk = a.bs_log2 >= 0 ? slot >> a.bs_log2 : slot / a.block_size;
    const int64_t row = slot - blk * a.block_size;
    const int h = a.hd_log2 >= 0 ? col >> a.hd_log2 : col / a.head_dim;
    const int e = col - h * a.head_dim;
    const int64_t dst = ((blk * a.num_kv_heads + h) * a.block_size + row) * a.head_dim + e;
    void* pool = is_v ? a.v_pool : a.k_pool;
    if (a.mode == kQkvBf16)
      static_cast<uint16_t*>(pool)[dst] = (uint16_t)bf16_rne(v);
    else
      static_cast<float*>(pool)[dst] = v;
    return;
  }
  a.y[(int64_t)r * a.cols + o] =
      a.mode == kResidual ? t.res + v : (a.mode == kGelu ? gelu_f(v) : v);
}

// Elements k .. k + 3 of a row of n floats without a branch: past the row's
// end it reads the row's start, which keep4 removes once the load has landed.
// VEC: the row is 16-byte aligned and n % 4 == 0.
template <bool VEC>
__device__ __forceinline__ f32x4_t load4(const float* p, int k, int n) {
  if constexpr (VEC) return *reinterpret_cast<const f32x4_t*>(p + (k < n ? k : 0));
  f32x4_t v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = p[k + e < n ? k + e : 0];
  return v;
}
// The same of four elements known to lie in the row.
template <bool VEC>
__device__ __forceinline__ f32x4_t load4u(const float* p) {
  if constexpr (VEC) return *reinterpret_cast<const f32x4_t*>(p);
  return f32x4_t{p[0], p[1], p[2], p[3]};
}
__device__ __forceinline__ f32x4_t keep4(const f32x4_t& v, int k, int n) {
  f32x4_t y;
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = k + e < n ? v[e] : 0.0f;
  return y;
}

// A barrier that orders LDS only: loads from global memory stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

constexpr int kChunk = 64;        // features per staged chunk
constexpr int kRow = kChunk + 4;  // LDS row stride: an odd count of 16-byte units,
                                  // so 16-byte reads of 64 rows hit distinct banks

// Layer-norm statistics (mean, sqrt(var + eps)) of the 4 NW rows of a
// workgroup to s_stat: the reference's two serial sums per row, whose 2 n
// dependent additions set the time.  Every wave loads (and squares) its four
// rows' terms, 16 lanes a row, kStat features at a time; they pass through LDS
// (buf: 2 x 4 NW rows of kStat + 4 floats) a piece ahead, and wave 0 adds them,
// a lane (or a quarter wave) a row, 16 reads a burst (a wave pays some 17 cycles to turn
// from additions to LDS reads).  64 tokens of Llama-3-8B's q / k / v: 141 us;
// every wave adding its own four rows reads LDS four times as often, 152;
// handing terms around with row_newbcast 171.
constexpr int kStat = 256;
template <bool VEC, int NW>
__device__ __forceinline__ void row_stats(const float* xr, int n, float eps, float* buf,
                                          float2* s_stat) {
#pragma clang fp contract(off)
  constexpr int ROWS = 4 * NW, S = kStat + 4, U = kStat / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, k4 = 4 * (lane & 15);
  const int slot = 4 * wave + (lane >> 4);  // the row this lane loads for
  float* wr = buf + slot * S + k4;
  // the row this lane adds: with one wave the one it loads, so that its mean
  // needs no exchange
  const int row = NW == 1 ? slot : lane & (ROWS - 1);
  const float* rd = buf + row * S;
  const int whole = n / kStat;
  auto pass = [&](auto term) __attribute__((always_inline)) {
    float acc = 0.0f;
    f32x4_t t[2][16];
    auto read = [&](f32x4_t(&d)[16], const float* b) __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < 16; ++s) d[s] = *reinterpret_cast<const f32x4_t*>(b + 4 * s);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto add = [&](const f32x4_t(&d)[16]) __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < 16; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = acc + d[s][e];
      __builtin_amdgcn_sched_barrier(0);
    };
    f32x4_t v[U];
    if (whole) {
      auto request = [&](int piece) __attribute__((always_inline)) {
        const float* p = xr + (piece < whole ? piece : whole - 1) * kStat + k4;
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = load4u<VEC>(p + 64 * u);
      };
      auto stage = [&](int i) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          *reinterpret_cast<f32x4_t*>(wr + i * ROWS * S + 64 * u) = term(v[u]);
      };
      request(0);
      stage(0);
      request(1);
      lds_barrier();
      for (int c = 0; c < whole; ++c) {
        stage((c + 1) & 1);  // the last round's is not added
        request(c + 2);
        if (wave == 0) {
          const float* b = rd + (c & 1) * ROWS * S;
          read(t[0], b);
          read(t[1], b + 64);
          add(t[0]);
          read(t[0], b + 128);
          add(t[1]);
          read(t[1], b + 192);
          add(t[0]);
          add(t[1]);
        }
        lds_barrier();
      }
    }
    const int k0 = whole * kStat;
    if (k0 < n) {  // features past the end add +0
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (k0 + 64 * u < n) v[u] = load4<VEC>(xr, k0 + 64 * u + k4, n);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (k0 + 64 * u < n)
          *reinterpret_cast<f32x4_t*>(wr + 64 * u) = keep4(term(v[u]), k0 + 64 * u + k4, n);
      lds_barrier();
      if (wave == 0) {
        const float* b = rd;
        for (int k = k0; k < n; k += 128, b += 128) {
          read(t[0], b);
          read(t[1], b + 64);
          add(t[0]);
          if (k + 64 < n) add(t[1]);
        }
      }
      lds_barrier();
    }
    return acc;
  };
  const float mean = pass([](const f32x4_t& x) { return x; }) / (float)n;
  float m = mean;
  if (wave == 0) s_stat[row].x = mean;  // every lane of a row the same
  if constexpr (NW > 1) {
    lds_barrier();
    m = s_stat[slot].x;
  }
  const float vs = pass([&](const f32x4_t& x) __attribute__((always_inline)) {
    f32x4_t t;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float d = x[e] - m;
      t[e] = d * d;
    }
    return t;
  });
  if (wave == 0) s_stat[row].y = sqrtf(vs / (float)n + eps);
  lds_barrier();
}

// Lane J of each row of 16 lanes, to the whole row.
template <int J>
__device__ __forceinline__ float row_bcast(float x) {
  return __int_as_float(
      __builtin_amdgcn_mov_dpp(__float_as_int(x), 0x150 + J /* row_newbcast */, 0xf, 0xf, true));
}

// A workgroup is NW waves on the same OW output columns; wave w owns rows
// RW w .. RW w + RW - 1 of the workgroup's NW * RW.  Lane l accumulates column
// l % OW of its wave's RW rows.
// RW = 4: per feature k one MFMA: B is the column's weight (lane l: w[l][k]),
// A the rows' features -- one 16-byte load per lane brings 64 features of the
// four rows (lane 4 j + i: row i, features 4 j .. + 3), and cbsz = 4 /
// abid = j hand the lanes of block j to all 16 blocks -- and result register e
// is row e of every column.  A group's MFMAs are issued before the additions
// of the group before, so no addition waits for its product (37 cycles a
// feature and four rows; alternating the two one by one is a quarter slower).
// RW = 1: lane j of each 16 holds features 4 j .. + 3 of the row and
// row_newbcast hands one to the multiplication.
// Weights pass through LDS, a chunk of 64 features in each of three buffers:
// chunk c + 1 is written early in chunk c, one barrier late in chunk c makes
// it visible and frees the buffer of chunk c - 1, so the steps run on across
// chunks; two more chunks are on their way in registers.
template <bool VEC, bool LN, int RW, int OW, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2))) void proj_kernel(
    ProjArgs a) {
#pragma clang fp contract(off)
  constexpr bool MFMA = RW == 4;
  // Groups of 4 GS features: a wave pays some 17 cycles for turning from vector
  // instructions to LDS reads and 10 for turning from MFMAs to additions, so
  // both go in groups.
  constexpr int GS = MFMA ? 2 : 4, NG = kChunk / 4 / GS;
  constexpr int NX = MFMA ? 1 : RW;  // x loads of a lane per chunk
  constexpr int NL = OW * (kChunk / 4) / (64 * NW);  // float4 of weights a thread stages
  static_assert(NL * 4 * NW == OW, "staging split");
  constexpr int WB = OW * kRow;  // floats of a weight buffer
  constexpr int SB = LN ? 8 * NW * (kStat + 4) : 0;  // floats of the statistics' buffers
  __shared__ __align__(16) float s_buf[3 * WB > SB ? 3 * WB : SB];
  __shared__ float2 s_stat[LN ? 4 * NW : 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = a.n;
  const int64_t o0 = ((int64_t)blockIdx.z * gridDim.x + blockIdx.x) * OW;
  if (o0 >= a.cols) return;  // the whole workgroup: the last row of a split grid
  const auto col = [&](int i) __attribute__((always_inline)) {  // column o0 + i, clamped
    return (int)(o0 + i < a.cols ? o0 + i : a.cols - 1);
  };
  const int r0 = (blockIdx.y * NW + wave) * RW;

  // staging: thread t takes float4 t % 16 of columns t / 16 + 4 NW i
  const int sk = 4 * (tid & 15), so = tid >> 4;
  const float* wrow[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) wrow[i] = weight_row(a, col(so + 4 * NW * i));
  const int pairs = n / (2 * kChunk) * 2;  // chunks the pipelined loop covers
  f32x4_t wv[2][NL];
  auto wload = [&](f32x4_t(&d)[NL], int chunk) __attribute__((always_inline)) {
    const int k = (chunk < pairs ? chunk : pairs - 1) * kChunk + sk;
#pragma unroll
    for (int i = 0; i < NL; ++i) d[i] = load4u<VEC>(wrow[i] + k);
  };
  auto wstore = [&](const f32x4_t(&d)[NL], float* buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NL; ++i)
      *reinterpret_cast<f32x4_t*>(buf + (so + 4 * NW * i) * kRow + sk) = d[i];
  };
  if (pairs) {
    wload(wv[0], 0);
    wload(wv[1], 1);
  }

  const auto row_of = [&](int i) __attribute__((always_inline)) {  // this wave's row i, clamped
    const int r = r0 + (i < RW ? i : 0);
    return a.x + (int64_t)(r < a.rows ? r : a.rows - 1) * n;
  };
  const int xk = 4 * (MFMA ? lane >> 2 : lane & 15);
  const float* xrow[NX];
#pragma unroll
  for (int i = 0; i < NX; ++i) xrow[i] = row_of(MFMA ? lane & 3 : i);
  f32x4_t xv[2][NX], gv[LN ? 2 : 1], bv[LN ? 2 : 1];
  auto xload = [&](int p, int chunk) __attribute__((always_inline)) {
    const int k = (chunk < pairs ? chunk : pairs - 1) * kChunk + xk;
#pragma unroll
    for (int i = 0; i < NX; ++i) xv[p][i] = load4u<VEC>(xrow[i] + k);
    if constexpr (LN) {
      gv[p] = load4u<VEC>(a.ln_g + k);
      bv[p] = load4u<VEC>(a.ln_b + k);
    }
  };
  if (pairs) {
    xload(0, 0);
    xload(1, 1);
  }
  // the output column and rows of this lane (duplicates and rows past the end
  // clamped: loaded, not stored)
  const int o = col(lane % OW);
  const ColTail ct = col_tail(a, o);
  RowTail rt[RW];
#pragma unroll
  for (int e = 0; e < RW; ++e) rt[e] = row_tail(a, r0 + e < a.rows ? r0 + e : a.rows - 1, o);
  float2 st[NX];
  if constexpr (LN) {
    row_stats<VEC, NW>(row_of(lane >> 4), n, a.eps, s_buf, s_stat);
#pragma unroll
    for (int i = 0; i < NX; ++i) st[i] = s_stat[4 * wave + (MFMA ? lane & 3 : i)];
    lds_barrier();  // the buffers become weights
  }
  float *cur = s_buf, *next = s_buf + WB, *spare = s_buf + 2 * WB;
  const int wl = (lane % OW) * kRow;  // this lane's column in a buffer
  const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
  float acc[RW];
#pragma unroll
  for (int e = 0; e < RW; ++e) acc[e] = 0.0f;
  f32x4_t p[2][4 * GS];  // RW = 4: products of the current and the previous group
#pragma unroll
  for (int c = 0; c < 4 * GS; ++c) p[1][c] = zero;
  f32x4_t wr[2][GS];  // weights of this group and the next
  auto read_w = [&](f32x4_t(&d)[GS], const float* b) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < GS; ++j) d[j] = *reinterpret_cast<const f32x4_t*>(b + wl + 4 * j);
  };
  // Chunk c: weights in cur, x in xv[I].  LOOP: the next chunks are on their
  // way (wv[I ^ 1] holds chunk c + 1's weights).
  auto chunk = [&](auto ic, auto loop, int c) __attribute__((always_inline)) {
    constexpr int I = decltype(ic)::value;
    constexpr bool LOOP = decltype(loop)::value;
    f32x4_t xa[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      xa[i] = xv[I][i];
      if constexpr (LN) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          xa[i][e] = (xa[i][e] - st[i].x) / st[i].y * gv[I][e] + bv[I][e];
      }
      if constexpr (!LOOP) xa[i] = keep4(xa[i], c * kChunk + xk, n);
    }
    if constexpr (LOOP) xload(I, c + 2);
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, NG>([&](auto gc) __attribute__((always_inline)) {
      constexpr int g = decltype(gc)::value;
      if constexpr (LOOP && g == 1) {
        wstore(wv[I ^ 1], next);
        wload(wv[I ^ 1], c + 3);
      }
      if constexpr (LOOP && g == NG - 1) lds_barrier();
      if constexpr (LOOP || g + 1 < NG)  // the next group's weights
        read_w(wr[(g + 1) & 1], g + 1 < NG ? cur + 4 * GS * (g + 1) : next);
      __builtin_amdgcn_sched_barrier(0);
      const f32x4_t(&w)[GS] = wr[g & 1];
      if constexpr (MFMA) {
        static_for<0, GS>([&](auto jc) __attribute__((always_inline)) {
          constexpr int j = decltype(jc)::value;
#pragma unroll
          for (int t = 0; t < 4; ++t)
            p[g & 1][4 * j + t] = __builtin_amdgcn_mfma_f32_4x4x1f32(xa[0][t], w[j][t], zero, 4,
                                                                     GS * g + j, 0);
        });
#pragma unroll
        for (int t = 0; t < 4 * GS; ++t)
#pragma unroll
          for (int e = 0; e < RW; ++e) acc[e] = acc[e] + p[(g & 1) ^ 1][t][e];
        __builtin_amdgcn_sched_group_barrier(0x008, 4 * GS, 0);       // the group's MFMAs,
        __builtin_amdgcn_sched_group_barrier(0x002, 4 * RW * GS, 0);  // then the additions
      } else {
        static_for<0, GS>([&](auto jc) __attribute__((always_inline)) {
          constexpr int j = decltype(jc)::value;
          float pr[RW][4];
#pragma unroll
          for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int e = 0; e < RW; ++e) pr[e][t] = row_bcast<GS * g + j>(xa[e][t]) * w[j][t];
#pragma unroll
          for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int e = 0; e < RW; ++e) acc[e] = acc[e] + pr[e][t];
        });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    float* const f = cur;
    cur = next, next = spare, spare = f;
  };
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  constexpr std::true_type looped{};
  constexpr std::false_type last{};
  if (pairs) {
    wstore(wv[0], cur);
    wload(wv[0], 2);
    lds_barrier();
    read_w(wr[0], cur);
    for (int c = 0; c < pairs; c += 2) {
      chunk(even, looped, c);
      chunk(odd, looped, c + 1);
    }
  }
  for (int c = pairs; c * kChunk < n; ++c) {  // at most two more, the last perhaps partial
    lds_barrier();                            // every wave has read its last chunk
#pragma unroll
    for (int i = 0; i < NL; ++i)
      wv[0][i] = keep4(load4<VEC>(wrow[i], c * kChunk + sk, n), c * kChunk + sk, n);
    wstore(wv[0], cur);
#pragma unroll
    for (int i = 0; i < NX; ++i) xv[0][i] = load4<VEC>(xrow[i], c * kChunk + xk, n);
    if constexpr (LN) {
      gv[0] = load4<VEC>(a.ln_g, c * kChunk + xk, n);
      bv[0] = load4<VEC>(a.ln_b, c * kChunk + xk, n);
    }
    lds_barrier();
    read_w(wr[0], cur);
    chunk(even, last, c);
  }
  if constexpr (MFMA) {
    // the last step's products: their additions stay clear of its MFMAs
    asm volatile("s_nop 7");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 4 * GS; ++t)
#pragma unroll
      for (int e = 0; e < RW; ++e) acc[e] = acc[e] + p[1][t][e];  // a chunk has an even count
  }

  if (lane < OW && o0 + lane < a.cols) {
#pragma unroll
    for (int e = 0; e < RW; ++e)
      if (r0 + e < a.rows) put(a, r0 + e, o, acc[e], ct, rt[e]);
  }
}

// Which split.  A wave computes 64 columns of one row (RW = 1) or of four
// (RW = 4), 16 columns of one row where the call is small.  Measured in us at
// n = 4,096 for 4,096 columns (the kernel before it, one thread per output with
// un-staged weights, in brackets), RW = 1 x 16 columns / 1 x 64 / 4 x 64:
//   1 row 27 / 36 / 64 [79], 4 rows 31 / 36 / 64 [79], 8 rows 43 / 36 / 64
//   [79], 16 rows 73 / 37 / 63 [128], 32 rows 139 / 53 / 64 [253], 48 rows 199
//   / 70 / 64 [377], 64 rows 255 / 90 / 64 [501], 256 rows 943 / 345 / 163
//   [2009].
// Time is set by the wave's serial chain while there is at most one wave per
// SIMD (1,024), then grows by 18 us a wave (RW = 1) or 36 us (RW = 4): the
// narrow split up to 1,024 of its waves, four rows a wave from 2,048 waves of
// one row on.  With the layer norm each workgroup also forms its rows' sums
// (37 us, for one row or sixteen): four rows a wave from 1,024 (11 rows of 6,144 columns
// 109 / 106, 16 rows 112 / 105; 8 rows 77 / 104; each some 3 to 10 less since
// one wave adds a workgroup's sums).
// Narrow calls of up to two rows take one-wave workgroups (1 row 27.3 against
// 31.7 us), others four rows a workgroup sharing the weights (8 x 8,192 x
// 1,024: 56.6 against 57.5).  One row takes them at any width, since three of
// four waves of a wider split have no row: 128,256 columns, 1 x 16 columns / 1 x
// 64 / 4 x 64 [before]: n = 4,096 380 / 428 / 451 [427], 512 42.7 / 43.1 / 51.1
// [45.4], 128 13.5 / 14.7 / 17.9 [13.3]; with the layer norm, 128,000 columns, n =
// 4,096 463 / 497 / 576 [618].
template <bool VEC, bool LN>
void launch(const ProjArgs& a, hipStream_t s) {
  auto go = [&](auto rw, auto ow, auto nw) {
    constexpr int RW = decltype(rw)::value, OW = decltype(ow)::value, NW = decltype(nw)::value;
    // a grid dimension times the workgroup stays under 2^32 threads
    const int64_t groups = ((int64_t)a.cols + OW - 1) / OW;
    const int64_t gx = groups < (1 << 22) ? groups : (1 << 22);
    const dim3 grid((unsigned)gx, (unsigned)((a.rows + RW * NW - 1) / (RW * NW)),
                    (unsigned)((groups + gx - 1) / gx));
    proj_kernel<VEC, LN, RW, OW, NW><<<grid, 64 * NW, 0, s>>>(a);
  };
  constexpr std::integral_constant<int, 1> c1{};
  constexpr std::integral_constant<int, 4> c4{};
  constexpr std::integral_constant<int, 16> c16{};
  constexpr std::integral_constant<int, 64> c64{};
  const int64_t rows = a.rows, rows4 = (rows + 3) / 4 * 4;
  const int64_t narrow = ((int64_t)a.cols + 15) / 16, wide = ((int64_t)a.cols + 63) / 64;
  if (rows == 1 || narrow * rows <= 1024)
    rows <= 2 ? go(c1, c16, c1) : go(c1, c16, c4);
  else if (wide * rows4 <= (LN ? 1024 : 2048))
    go(c1, c64, c4);
  else
    go(c4, c64, c4);
}

int dispatch(const ProjArgs& a, bool w_aligned, hipStream_t s, const char* what) {
  const bool vec = w_aligned && a.n % 4 == 0 && aligned16(a.x) &&
                   (!a.ln_g || (aligned16(a.ln_g) && aligned16(a.ln_b)));
  if (vec)
    a.ln_g ? launch<true, true>(a, s) : launch<true, false>(a, s);
  else
    a.ln_g ? launch<false, true>(a, s) : launch<false, false>(a, s);
  return check_launch(what);
}

constexpr int kMaxIn = 8192;  // input features the entry points accept

}  // namespace

// Shared by rkv_linear and the decoder / engine (fused epilogues).
int linear_launch(float* y, const float* x, const float* w, const float* b, const float* res,
                  int epi, int rows, int in_dim, int out_dim, hipStream_t s, const float* ln_g,
                  const float* ln_b, float eps) {
  if (rows < 0 || in_dim <= 0 || out_dim <= 0)
    return fail(RKV_ERR_INVALID_ARG, "rkv_linear: bad size argument");
  if (rows == 0) return RKV_OK;
  if (rows > 65535) return fail(RKV_ERR_INVALID_ARG, "rkv_linear: rows must be <= 65535");
  if (in_dim > kMaxIn) return fail(RKV_ERR_UNSUPPORTED, "rkv_linear: in_dim must be <= 8192");
  if (!y || !x || !w || (epi == 1 && !res))
    return fail(RKV_ERR_INVALID_ARG, "rkv_linear: null pointer argument");
  if (!ln_g != !ln_b) return fail(RKV_ERR_INVALID_ARG, "rkv_linear: ln_g and ln_b go together");
  ProjArgs a{};
  a.y = y, a.x = x, a.w = w, a.b = b, a.res = res, a.ln_g = ln_g, a.ln_b = ln_b, a.eps = eps;
  a.rows = rows, a.n = in_dim, a.cols = out_dim;
  a.mode = epi == 1 ? kResidual : (epi == 2 ? kGelu : kPlain);
  return dispatch(a, aligned16(w), s, "rkv_linear");
}

}  // namespace rkv

using namespace rkv;

extern "C" int rkv_linear(float* y, const float* x, const float* w, const float* b, int rows,
                          int in_dim, int out_dim, void* stream) {
  clear_error();
  return linear_launch(y, x, w, b, nullptr, 0, rows, in_dim, out_dim,
                       static_cast<hipStream_t>(stream));
}

extern "C" int rkv_qkv_append(float* q_out, void* k_pool, void* v_pool,
                              const int64_t* slot_mapping, const float* x, const float* ln_g,
                              const float* ln_b, float eps, const float* wq, const float* bq,
                              const float* wk, const float* bk, const float* wv,
                              const float* bv, int n_tokens, int d_model, int q_dim,
                              int num_kv_heads, int head_dim, int block_size,
                              int64_t num_blocks, int dtype, void* stream) {
  clear_error();
  if (n_tokens < 0 || d_model <= 0 || q_dim <= 0 || num_kv_heads <= 0 || head_dim <= 0 ||
      block_size <= 0 || num_blocks <= 0)
    return fail(RKV_ERR_INVALID_ARG, "rkv_qkv_append: bad size argument");
  if (d_model > kMaxIn)
    return fail(RKV_ERR_UNSUPPORTED, "rkv_qkv_append: d_model must be <= 8192");
  if (n_tokens > 65535)
    return fail(RKV_ERR_INVALID_ARG, "rkv_qkv_append: n_tokens must be <= 65535");
  if ((int64_t)q_dim + 2 * (int64_t)num_kv_heads * head_dim > (int64_t)INT32_MAX - 64)
    return fail(RKV_ERR_INVALID_ARG, "rkv_qkv_append: too many output columns");
  if (dtype != RKV_F32 && dtype != RKV_BF16)
    return fail(RKV_ERR_UNSUPPORTED, "rkv_qkv_append: pools must be RKV_F32 or RKV_BF16");
  if (!ln_g != !ln_b)
    return fail(RKV_ERR_INVALID_ARG, "rkv_qkv_append: ln_g and ln_b are both given or both NULL");
  if (n_tokens == 0) return RKV_OK;
  if (!q_out || !k_pool || !v_pool || !slot_mapping || !x || !wq || !wk || !wv)
    return fail(RKV_ERR_INVALID_ARG, "rkv_qkv_append: null pointer argument");
  ProjArgs a{};
  a.y = q_out, a.x = x, a.w = wq, a.b = bq, a.ln_g = ln_g, a.ln_b = ln_b, a.eps = eps;
  a.wk = wk, a.bk = bk, a.wv = wv, a.bv = bv, a.k_pool = k_pool, a.v_pool = v_pool;
  a.slots = slot_mapping, a.num_slots = num_blocks * block_size;
  a.q_dim = q_dim, a.kvd = num_kv_heads * head_dim;
  a.num_kv_heads = num_kv_heads, a.head_dim = head_dim, a.block_size = block_size;
  const auto log2_of = [](int v) { return (v & (v - 1)) == 0 ? __builtin_ctz(v) : -1; };
  a.hd_log2 = log2_of(head_dim), a.bs_log2 = log2_of(block_size);
  a.rows = n_tokens, a.n = d_model, a.cols = q_dim + 2 * a.kvd;
  a.mode = dtype == RKV_BF16 ? kQkvBf16 : kQkvF32;
  return dispatch(a, aligned16(wq) && aligned16(wk) && aligned16(wv),
                  static_cast<hipStream_t>(stream), "rkv_qkv_append");
}
