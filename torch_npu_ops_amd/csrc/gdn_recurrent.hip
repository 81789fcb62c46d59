// Gated delta rule, recurrent form (decode / short speculative windows),
// and the decode step fused with the causal conv1d update, for gfx950.
//
// Per token (reference kernel triton_npu/triton_src/
// test_fused_recurrent_gated_delta_rule.py:125-164, CPU golden
// triton_npu/test/triton_recurrent_gated_delta_rule_test.cpp:47-115):
//   q, k <- q/sqrt(sum q^2 + 1e-6), k/sqrt(sum k^2 + 1e-6)   (if l2norm)
//   q    <- q * scale
//   h    <- exp(g) * h                       h: [K, V] fp32 per (slot, head)
//   v'   <- beta * (v - h^T k)
//   h    <- h + k v'^T
//   o    <- h^T q
// GQA: v-head hv reads qk-head hv / (HV / H).  State slots come from
// ssm_state_indices; with num_accepted_tokens (speculative decoding) the
// initial state is column accepted-1 and the state after token t goes to
// column t (..._spec_fwd_kernel, :257-307).
//
// Design (HBM-bound state streaming): one 256-lane block per (sequence,
// v-head) keeps the whole K x V fp32 state in registers, K*V/256 values per
// lane laid out so that each row of V values is contiguous across V/4
// lanes (16-byte accesses, 1 KB per wave per instruction).  h^T k and h^T q
// of the decayed state come out of one pass over the registers and one
// cross-wave LDS reduction (o = (e^g h)^T q + (k.q) v', so the update and
// the output need no second pass); the rank-1 update is applied in
// registers and the state is written back once.  State traffic uses
// non-temporal hints: it is read and written exactly once per call.  A token
// takes one barrier (gdn_token); a decode layer's step for one sequence of 32
// v-heads, replayed from a graph on MI355X, went from 24.1 to 22.9 us with
// that (six barriers before), large batches stay at the state stream's rate.
#include "xk_common.h"

namespace xk {
namespace {

constexpr int kThreads = 256;
// The fused decode kernel keeps one block per (batch row, qk head) and
// spreads each 64 KB state tile over 512 lanes (8 loads per lane): an
// in-place stream of 64 KB tiles runs at 5.5 TB/s on MI355X with 16 loads
// per lane, at 6.2 TB/s with 8.
constexpr int kFusedThreads = 512;

// Per-lane share of a K x V state tile.
template <int K, int V, int NT = kThreads>
struct Tile {
  static constexpr int kLanesPerRow = V / 4;               // float4 per lane
  static constexpr int kRowsPerPass = NT / kLanesPerRow;
  static constexpr int kPasses = K / kRowsPerPass;
  static_assert(V % 4 == 0 && kLanesPerRow <= kWave && kWave % kLanesPerRow == 0,
                "row of V must fit a wave");
  static_assert(K % kRowsPerPass == 0, "K must be a multiple of rows per pass");
  float h[kPasses][4];
};

// Per-wave partials of h^T k and h^T q, double-buffered from one token (or
// head) to the next: written before a token's barrier, read until the next
// one's.
template <int V, int NT = kThreads>
struct Partials {
  float p[2][2][NT / kWave][V];
};

template <typename T>
__device__ __forceinline__ float ldf(const void* p, int64_t i) {
  return to_f32(reinterpret_cast<const T*>(p)[i]);
}

// softplus(x) = max(x, 0) + log1p(e^-|x|) on the hardware exp2 / log2
// (v_exp_f32, v_log_f32).  e^-|x| = 2^p (1 + p_lo ln 2) with p = fl(-|x|
// log2 e) and p_lo its rounding error (one fma) plus the error of the
// float log2 e, so the result stays within a few ulp for large |x| too;
// log1p(u) = log(1 + u) * u / ((1 + u) - 1) (Goldberg's correction; (1 + u)
// - 1 is exact, and 1 + u == 1 gives u).  About 20 instructions against
// ~100 for log1pf(expf(x)).
__device__ __forceinline__ float softplus_hw(float x) {
  constexpr float kLog2e = 1.44269502162933349609375f;  // float(log2 e)
  constexpr float kLog2eLo = 1.925963e-08f;              // log2 e - kLog2e
  constexpr float kLn2 = 0.693147180559945309f;
  const float t = -fabsf(x);
  const float p = t * kLog2e;
  const float plo = fmaf(t, kLog2e, -p) + t * kLog2eLo;
  const float u0 = __builtin_amdgcn_exp2f(p);
  const float u = fmaf(u0, plo * kLn2, u0);
  const float w = 1.f + u;
  const float d = w - 1.f;
  const float lp = d == 0.f ? u : __builtin_amdgcn_logf(w) * kLn2 * (u * __builtin_amdgcn_rcpf(d));
  return fmaxf(x, 0.f) + lp;
}

// GDN gating (triton_src/test_fused_gdn_gating.py:30-43): the log-decay
// g = -exp(A_log) * softplus_{beta, threshold}(a + dt_bias), where softplus
// is log(1 + exp(beta x)) / beta below the threshold and x above it.  Both
// exponentials use the hardware exp2 (exp(A_log) to ~1e-7 |A_log|
// relative): g is fp32 and the reference's test holds it to rtol / atol
// 1e-3 (test_fused_gdn_gating.py:107); the error here is below 1e-6.
// inv_beta is 1 / sp_beta, multiplied in as the reference does.
__device__ __forceinline__ float gdn_log_decay(float a_plus_bias, float A_log, float sp_beta,
                                               float inv_beta, float threshold) {
  constexpr float kLog2e = 1.44269504088896341f;
  const float bx = sp_beta * a_plus_bias;
  const float sp = bx <= threshold ? inv_beta * softplus_hw(bx) : a_plus_bias;
  return -__builtin_amdgcn_exp2f(A_log * kLog2e) * sp;
}

// sigmoid with IEEE division and the accurate exp, so that a rounded
// 16-bit result matches a CPU computation of the same expression.
__device__ __forceinline__ float sigmoid_exact(float x) { return 1.0f / (1.0f + expf(-x)); }

// sigmoid(x) rounded to bf16, equal to sigmoid_exact's rounding.  For
// |x| < 32 the hardware exp2 / rcp value is within about 50 fp32 ulp of
// sigmoid_exact's: fl(-x log2 e) (< 64 in magnitude) is off by at most
// 2^-19 for its rounding plus 32 * 2^-24 for the float log2 e, i.e. 2^-18,
// which is 44 ulp of exp2 at most; exp2, the add, rcp and sigmoid_exact
// itself add a few more.  So when the fast value's low 16 bits are more than
// 128 from the bf16 rounding boundary 0x8000, both round to the same bf16.
// Elsewhere (0.4% of values, and |x| >= 32 or NaN) sigmoid_exact is used.
__device__ __forceinline__ bf16 sigmoid_bf16(float x) {
  constexpr float kLog2e = 1.44269504088896341f;
  float s = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-x * kLog2e));
  const uint32_t low = __builtin_bit_cast(uint32_t, s) & 0xFFFFu;
  if (!(fabsf(x) < 32.f) || (low > 0x8000u - 128u && low < 0x8000u + 128u)) s = sigmoid_exact(x);
  return from_f32<bf16>(s);
}

template <typename AB>
__device__ __forceinline__ AB sigmoid_to(float x) {
  if constexpr (std::is_same<AB, bf16>::value) {
    return sigmoid_bf16(x);
  } else {
    return from_f32<AB>(sigmoid_exact(x));
  }
}

// Sum over the lanes of a wave that differ in lane bits 4 and 5 (STAGE 16 and
// 32), by swapping 16-lane rows / wave halves of two copies of the value.
template <int STAGE>
__device__ __forceinline__ float swap_sum(float v) {
  static_assert(STAGE == 16 || STAGE == 32, "row or half");
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  typedef unsigned int u2_t __attribute__((ext_vector_type(2)));
  u2_t r;
  if constexpr (STAGE == 16) r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  else r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const uint32_t x = r[0], y = r[1];  // (a bit cast of a vector element reads element 0)
  return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}

// 1 / sqrt(x) for x >= 1e-6: the hardware's estimate and one Newton step, as
// exact as 1.0f / sqrtf(x) in a fifth of its instructions (0 for +inf).  Every
// wave forms two of these a token, which a full chip is short of issue slots
// for: 8 tokens of 16 sequences x 32 v-heads (4 blocks on every CU) 27.1 us
// with the IEEE sequences, 25.2 with this, 26.2 when one wave formed them.
__device__ __forceinline__ float inv_sqrt(float x) {
  const float y = rsqrt_hw(x), z = fmaf(0.5f * y, fmaf(-x * y, y, 1.f), y);
  return x < __builtin_inff() ? z : y;
}

// Scalars of one token's q and k (raw, fp32, in LDS): rk = 1 / ||k||, rq =
// scale / ||q|| (norms with the 1e-6 of the l2norm; 1 without it) and kq =
// rk rq (k . q).  Every wave forms them for itself, so no barrier is needed
// between them and their use.
struct QkScales {
  float rk, rq, kq;
};
template <int K>
__device__ __forceinline__ QkScales qk_scales(const float* q, const float* k, bool l2norm,
                                              float scale) {
  const int lane = threadIdx.x % kWave;
  float sq = 0.f, sk = 0.f, kq = 0.f;
#pragma unroll
  for (int i = lane; i < K; i += kWave) {
    const float qv = q[i], kv = k[i];
    sq = fmaf(qv, qv, sq);
    sk = fmaf(kv, kv, sk);
    kq = fmaf(qv, kv, kq);
  }
  sq = group_sum<kWave>(sq);
  sk = group_sum<kWave>(sk);
  kq = group_sum<kWave>(kq);
  QkScales r;
  r.rk = l2norm ? inv_sqrt(sk + 1e-6f) : 1.0f;
  r.rq = (l2norm ? inv_sqrt(sq + 1e-6f) : 1.0f) * scale;
  r.kq = kq * r.rk * r.rq;
  return r;
}

// One token of the recurrence on the register tile, with one barrier.  q, k
// and v (raw, fp32, LDS) were complete at the barrier before; `before` runs
// ahead of this one's barrier (it may fill the other input buffer) and
// store_o(column, four outputs) is called by the lanes of the first row.
// Every lane sums the waves' partials of its own four columns after the
// barrier and applies the norms of q and k as scalars, where writing
// normalised q and k, then v', back through LDS took five more barriers.
template <int K, int V, int NT, typename Before, typename StoreO>
__device__ __forceinline__ void gdn_token(Tile<K, V, NT>& t, Partials<V, NT>& red, int buf,
                                          const float* q, const float* k, const float* v,
                                          const QkScales& sc, float decay, float beta,
                                          Before before, StoreO store_o) {
  using TL = Tile<K, V, NT>;
  const int tid = threadIdx.x;
  const int c4 = tid % TL::kLanesPerRow;  // column group (4 columns)
  const int r0 = tid / TL::kLanesPerRow;  // first row
  const int wid = tid / kWave;
  float pk[4] = {0.f, 0.f, 0.f, 0.f}, pq[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < TL::kPasses; ++i) {
    const int r = r0 + i * TL::kRowsPerPass;
    const float kr = k[r], qr = q[r];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      t.h[i][c] *= decay;
      pk[c] = fmaf(t.h[i][c], kr, pk[c]);
      pq[c] = fmaf(t.h[i][c], qr, pq[c]);
    }
  }
  // Reduce over the rows held by the other lanes of this wave (same c4).
  static_assert(TL::kLanesPerRow == 16 || TL::kLanesPerRow == 32, "rows of 64 or 128 columns");
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if constexpr (TL::kLanesPerRow == 16) {
      pk[c] = swap_sum<16>(pk[c]);
      pq[c] = swap_sum<16>(pq[c]);
    }
    pk[c] = swap_sum<32>(pk[c]);
    pq[c] = swap_sum<32>(pq[c]);
  }
  typedef Vec<float, 4> V4;
  if ((tid % kWave) < TL::kLanesPerRow) {
    *reinterpret_cast<V4*>(&red.p[buf][0][wid][c4 * 4]) = V4{{pk[0], pk[1], pk[2], pk[3]}};
    *reinterpret_cast<V4*>(&red.p[buf][1][wid][c4 * 4]) = V4{{pq[0], pq[1], pq[2], pq[3]}};
  }
  before();
  __syncthreads();
  float a[4] = {0.f, 0.f, 0.f, 0.f}, b[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < NT / kWave; ++w) {
    const V4 x = *reinterpret_cast<const V4*>(&red.p[buf][0][w][c4 * 4]);
    const V4 y = *reinterpret_cast<const V4*>(&red.p[buf][1][w][c4 * 4]);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      a[c] += x.v[c];
      b[c] += y.v[c];
    }
  }
  const V4 vv = *reinterpret_cast<const V4*>(&v[c4 * 4]);
  float vn[4], o[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    // v' = beta (v - h^T k);  o = h^T q + (k.q) v'
    const float n = beta * (vv.v[c] - sc.rk * a[c]);
    o[c] = fmaf(sc.rq, b[c], sc.kq * n);
    vn[c] = sc.rk * n;
  }
  if (r0 == 0) store_o(c4 * 4, o);
#pragma unroll
  for (int i = 0; i < TL::kPasses; ++i) {
    const float kr = k[r0 + i * TL::kRowsPerPass];
#pragma unroll
    for (int c = 0; c < 4; ++c) t.h[i][c] = fmaf(kr, vn[c], t.h[i][c]);
  }
}

template <int K, int V, int NT>
// `pitch`: floats between rows in memory (the tile may be a column slice of
// a wider state).
__device__ __forceinline__ void load_tile(Tile<K, V, NT>& t, const float* base, int64_t pitch = V) {
  using TL = Tile<K, V, NT>;
  const int c4 = threadIdx.x % TL::kLanesPerRow;
  const int r0 = threadIdx.x / TL::kLanesPerRow;
#pragma unroll
  for (int i = 0; i < TL::kPasses; ++i) {
    const Vec<float, 4> v = ld_stream(reinterpret_cast<const Vec<float, 4>*>(
        base + static_cast<int64_t>(r0 + i * TL::kRowsPerPass) * pitch + c4 * 4));
#pragma unroll
    for (int c = 0; c < 4; ++c) t.h[i][c] = v.v[c];
  }
}

template <int K, int V, int NT>
__device__ __forceinline__ void zero_tile(Tile<K, V, NT>& t) {
#pragma unroll
  for (int i = 0; i < Tile<K, V, NT>::kPasses; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c) t.h[i][c] = 0.f;
}

template <int K, int V, int NT>
__device__ __forceinline__ void store_tile(const Tile<K, V, NT>& t, float* base, int64_t pitch = V) {
  using TL = Tile<K, V, NT>;
  const int c4 = threadIdx.x % TL::kLanesPerRow;
  const int r0 = threadIdx.x / TL::kLanesPerRow;
#pragma unroll
  for (int i = 0; i < TL::kPasses; ++i) {
    Vec<float, 4> v;
#pragma unroll
    for (int c = 0; c < 4; ++c) v.v[c] = t.h[i][c];
    st_stream(reinterpret_cast<Vec<float, 4>*>(
                  base + static_cast<int64_t>(r0 + i * TL::kRowsPerPass) * pitch + c4 * 4),
              v);
  }
}

// ---------------------------------------------------------------------------
// Recurrent GDN over varlen sequences.
// ---------------------------------------------------------------------------
struct RecParams {
  const void* q;
  const void* k;
  const void* v;
  int64_t sq, sk, sv;  // token pitches of q, k, v (elements); heads dense within a token
  const void* g;
  const void* beta;
  void* o;
  const float* h0;
  float* ht;
  int64_t h0_slot_stride, ht_slot_stride;
  int64_t slots;  // rows of the state pool (valid slot range)
  const void* cu;
  int cu_i64;
  const int32_t* idx;
  int64_t idx_s0, idx_s1;
  const int32_t* accepted;
  int64_t N, T;  // sequences; tokens per sequence when cu == NULL
  int H, HV;
  float scale;
  int l2norm;
  int inplace;
  // Gating mode: g holds a and beta holds b ([tokens, HV]); per token
  // g = gdn_log_decay(a + dt_bias, A_log), beta = sigmoid(b).
  int gating;
  const float* A_log;
  const float* dt_bias;
  float sp_beta, sp_thr;
};

// NS blocks per (sequence, v head), each owning VT = V / NS state columns
// (the recurrence is independent per column; q / k normalisation is
// repeated per block).  At V = 128, NS = 2: an in-place stream of 64 KB
// tiles with 16 loads per lane runs at 5.5 TB/s on MI355X, of 32 KB tiles
// with 8 loads per lane at 6.3 TB/s.
template <int K, int V, typename T, typename GT, typename BT, int NS>
__global__ void __launch_bounds__(kThreads) gdn_recurrent_kernel(RecParams p) {
  constexpr int VT = V / NS;
  // Raw inputs of a token.  A wave reads token i's until it reaches the
  // barrier of token i + 1, and those of token i + 1 are written before the
  // barrier of token i: three buffers.
  __shared__ __align__(16) struct {
    float q[3][K], k[3][K], v[3][VT];
  } in;
  __shared__ __align__(16) Partials<VT> red;
  const int cs = static_cast<int>(blockIdx.x % NS);  // column slice
  const int64_t item = blockIdx.x / NS;
  const int64_t n = item / p.HV;
  const int hv = static_cast<int>(item % p.HV);
  const int hq = hv / (p.HV / p.H);
  int64_t bos, len;
  if (p.cu) {
    const int64_t a = p.cu_i64 ? reinterpret_cast<const int64_t*>(p.cu)[n]
                               : reinterpret_cast<const int32_t*>(p.cu)[n];
    const int64_t b = p.cu_i64 ? reinterpret_cast<const int64_t*>(p.cu)[n + 1]
                               : reinterpret_cast<const int32_t*>(p.cu)[n + 1];
    bos = a;
    len = b - a;
  } else {
    bos = n * p.T;
    len = p.T;
  }
  if (len <= 0) return;  // whole block exits together

  const int64_t first_col = p.accepted ? p.accepted[n] - 1 : 0;
  auto slot_of = [&](int64_t col) -> int64_t {
    return p.idx ? p.idx[n * p.idx_s0 + col * p.idx_s1] : n;
  };
  // One token's inputs: lane tid holds element tid of q, k (tid < K) and v
  // (tid < V), plus the head's g and beta.
  const int tid = threadIdx.x;
  struct TokIn {
    float q, k, v, g, b;
  };
  auto load_in = [&](int64_t tok) {
    TokIn r;
    r.q = tid < K ? ldf<T>(p.q, tok * p.sq + hq * K + tid) : 0.f;
    r.k = tid < K ? ldf<T>(p.k, tok * p.sk + hq * K + tid) : 0.f;
    r.v = tid < VT ? ldf<T>(p.v, tok * p.sv + hv * V + cs * VT + tid) : 0.f;
    r.g = ldf<GT>(p.g, tok * p.HV + hv);
    r.b = p.beta ? ldf<BT>(p.beta, tok * p.HV + hv) : 1.0f;
    if (p.gating) {
      r.g = gdn_log_decay(r.g + p.dt_bias[hv], p.A_log[hv], p.sp_beta, 1.0f / p.sp_beta,
                          p.sp_thr);
      r.b = sigmoid_exact(r.b);
    }
    return r;
  };
  // The first token's inputs are fetched before the state tile: loads
  // complete in issue order, so the q/k normalisation then overlaps the
  // tile's latency instead of waiting behind it.
  TokIn cur = load_in(bos);
  Tile<K, VT> t;
  const int64_t s0 = slot_of(first_col);
  const bool s0_ok = p.h0 && s0 >= 0 && s0 < p.slots && first_col >= 0;
  const int64_t col0 = static_cast<int64_t>(hv) * K * V + cs * VT;  // slice within a slot
  if (s0_ok)
    load_tile<K, VT>(t, p.h0 + s0 * p.h0_slot_stride + col0, V);
  else
    zero_tile<K, VT>(t);

  // Per-token state writes: in place with a per-token slot column (2-D
  // indices or speculative decoding); otherwise once at the end.
  const bool per_token = p.inplace && p.idx && p.idx_s1 != 0;
  auto put = [&](int buf, const TokIn& r) {
    if (tid < K) {
      in.q[buf][tid] = r.q;
      in.k[buf][tid] = r.k;
    }
    if (tid < VT) in.v[buf][tid] = r.v;
  };
  put(0, cur);
  __syncthreads();
  int buf = 0;
  for (int64_t i = 0; i < len; ++i) {
    const int64_t tok = bos + i;
    const int next_buf = buf == 2 ? 0 : buf + 1;
    // The next token's inputs are fetched while this one computes, and put in
    // the next buffer ahead of this one's barrier.
    const TokIn nxt = i + 1 < len ? load_in(tok + 1) : cur;
    const QkScales sc = qk_scales<K>(in.q[buf], in.k[buf], p.l2norm, p.scale);
    T* o = reinterpret_cast<T*>(p.o) + (tok * p.HV + hv) * V + cs * VT;
    gdn_token<K, VT>(
        t, red, static_cast<int>(i & 1), in.q[buf], in.k[buf], in.v[buf], sc, __expf(cur.g), cur.b,
        [&]() { put(next_buf, nxt); },
        [&](int c, const float (&val)[4]) {
#pragma unroll
          for (int u = 0; u < 4; ++u) o[c + u] = from_f32<T>(val[u]);
        });
    // The block's waves write their rows of the state together: spread out,
    // the write stream costs 2% (182.9 against 186.7 us at batch 256).
    if (per_token) {
      __syncthreads();
      const int64_t sl = slot_of(i);
      if (sl >= 0 && sl < p.slots) store_tile<K, VT>(t, p.ht + sl * p.ht_slot_stride + col0, V);
    }
    cur = nxt;
    buf = next_buf;
  }
  if (!per_token) {
    __syncthreads();
    if (p.inplace) {
      if (s0 >= 0 && s0 < p.slots && first_col >= 0)
        store_tile<K, VT>(t, p.ht + s0 * p.ht_slot_stride + col0, V);
    } else {
      store_tile<K, VT>(t, p.ht + n * p.ht_slot_stride + col0, V);
    }
  }
}

template <int K, int V, typename T, typename GT>
int rec_beta(const RecParams& p, xk_dtype bdt, hipStream_t s) {
  constexpr int NS = V == 128 ? 2 : 1;  // column slices per (sequence, head)
  const dim3 grid(p.N * p.HV * NS);
  switch (bdt) {
    case XK_F32: hipLaunchKernelGGL((gdn_recurrent_kernel<K, V, T, GT, float, NS>), grid, dim3(kThreads), 0, s, p); break;
    case XK_BF16: hipLaunchKernelGGL((gdn_recurrent_kernel<K, V, T, GT, bf16, NS>), grid, dim3(kThreads), 0, s, p); break;
    case XK_F16: hipLaunchKernelGGL((gdn_recurrent_kernel<K, V, T, GT, f16, NS>), grid, dim3(kThreads), 0, s, p); break;
    default: return XK_ERR_UNSUPPORTED;
  }
  return launch_status();
}

template <int K, int V, typename T>
int rec_g(const RecParams& p, xk_dtype gdt, xk_dtype bdt, hipStream_t s) {
  switch (gdt) {
    case XK_F32: return rec_beta<K, V, T, float>(p, bdt, s);
    case XK_BF16: return rec_beta<K, V, T, bf16>(p, bdt, s);
    case XK_F16: return rec_beta<K, V, T, f16>(p, bdt, s);
    default: return XK_ERR_UNSUPPORTED;
  }
}

template <int K, int V>
int rec_t(const RecParams& p, xk_dtype dt, xk_dtype gdt, xk_dtype bdt, hipStream_t s) {
  switch (dt) {
    case XK_BF16: return rec_g<K, V, bf16>(p, gdt, bdt, s);
    case XK_F16: return rec_g<K, V, f16>(p, gdt, bdt, s);
    case XK_F32: return rec_g<K, V, float>(p, gdt, bdt, s);
    default: return XK_ERR_UNSUPPORTED;
  }
}

// ---------------------------------------------------------------------------
// GDN gating, elementwise over [rows, heads], one element per lane (the
// most lanes in flight: every wave makes one load-compute-store pass, so the
// compute is on each wave's critical path and more elements per lane only
// lengthen it).  IT is the index type: 32-bit below 2^31 elements.
// ---------------------------------------------------------------------------
constexpr int kGateBlock = 128;  // 3.20 us at the bench shape, 3.23 with 256

template <typename AB, typename IT>
__global__ void __launch_bounds__(kGateBlock)
    gdn_gating_kernel(const float* __restrict__ A_log, const AB* __restrict__ a,
                      const AB* __restrict__ b, const float* __restrict__ dt_bias,
                      float* __restrict__ g, AB* __restrict__ beta_out, IT n, int heads,
                      float sp_beta, float inv_beta, float threshold) {
  const IT i = static_cast<IT>(blockIdx.x) * kGateBlock + static_cast<IT>(threadIdx.x);
  if (i >= n) return;
  const AB av = ld_stream(a + i);
  const AB bv = ld_stream(b + i);
  // A power-of-two head count (the common case) is a mask, not a division.
  const int h = (heads & (heads - 1)) == 0 ? static_cast<int>(i & static_cast<IT>(heads - 1))
                                           : static_cast<int>(i % static_cast<IT>(heads));
  st_stream(g + i, gdn_log_decay(to_f32(av) + dt_bias[h], A_log[h], sp_beta, inv_beta, threshold));
  st_stream(beta_out + i, sigmoid_to<AB>(to_f32(bv)));
}

// ---------------------------------------------------------------------------
// Decode step fused with the conv1d update.  One block per (batch row,
// qk-head): it owns the conv channels of that q head, that k head and the
// HV/H v heads of the group, so every conv channel and every state tile is
// read and written by exactly one block.
// ---------------------------------------------------------------------------
struct FusedParams {
  const void* x;  // mixed_qkv [B, D] (D = 2*H*K + HV*V)
  int64_t sx;
  void* conv_state;  // [lines, D, S]
  int64_t cs_line, cs_dim, cs_tok;
  int64_t conv_lines;
  int S;  // conv state_len
  const void* w;  // [D, W]
  int64_t w_dim, w_tap;
  const void* cbias;  // [D] or NULL
  xk_dtype wdt;
  const int32_t* conv_idx;
  int W;
  const void* g;  // [B, HV]
  const void* beta;
  float* state;  // [slots, HV, K, V]
  int64_t st_slot_stride;
  int64_t slots;
  const int32_t* ssm_idx;
  void* o;  // [B, HV, V]
  int64_t B;
  int H, HV;
  float scale;
  int l2norm;
  int32_t pad;
  // Conv state [lines, D, S] with S contiguous per channel and lines 16-byte
  // aligned, weights [D, W] contiguous in x's dtype, W - 1 == S <= 8: eight
  // channels per lane with 16-byte loads and stores.
  int conv_vec;
  // Gating mode: g holds a and beta holds b ([B, HV]); g = gdn_log_decay(a +
  // dt_bias, A_log) and beta = sigmoid(b), per head, in registers.
  int gating;
  const float* A_log;
  const float* dt_bias;
  float sp_beta, sp_thr;
};

// Conv update + SiLU of 8 consecutive channels c0..c0+7 of batch row b
// (FusedParams::conv_vec layout); writes the shifted state back.
template <typename T, int S>
__device__ __forceinline__ void conv8(const FusedParams& p, int64_t b, int64_t cslot,
                                      bool conv_ok, int64_t c0, float (&y)[8]) {
  using V8 = Vec<T, 8>;
  constexpr int W = S + 1;
  const V8 xv = ld_stream(reinterpret_cast<const V8*>(reinterpret_cast<const T*>(p.x) +
                                                      b * p.sx + c0));
  Arr<T, 8 * W> wv;  // weights of the 8 channels, channel-major
#pragma unroll
  for (int q = 0; q < W; ++q)
    *reinterpret_cast<V8*>(&wv.v[8 * q]) =
        reinterpret_cast<const V8*>(reinterpret_cast<const T*>(p.w) + c0 * W)[q];
  Arr<T, 8 * S> sv;  // state of the 8 channels, channel-major
  T* st = reinterpret_cast<T*>(p.conv_state) + cslot * p.cs_line + c0 * S;
  if (conv_ok) {
#pragma unroll
    for (int q = 0; q < S; ++q)
      *reinterpret_cast<V8*>(&sv.v[8 * q]) = ld_stream(reinterpret_cast<const V8*>(st) + q);
  } else {
#pragma unroll
    for (int e = 0; e < 8 * S; ++e) sv.v[e] = from_f32<T>(0.f);
  }
  Arr<T, 8 * S> ns;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    float acc = p.cbias ? load_as_f32(p.cbias, c0 + c, p.wdt) : 0.f;
#pragma unroll
    for (int j = 0; j < S; ++j) acc = fmaf(to_f32(sv.v[c * S + j]), to_f32(wv.v[c * W + j]), acc);
    acc = fmaf(to_f32(xv.v[c]), to_f32(wv.v[c * W + S]), acc);
    y[c] = silu(acc);
#pragma unroll
    for (int j = 0; j + 1 < S; ++j) ns.v[c * S + j] = sv.v[c * S + j + 1];
    ns.v[c * S + S - 1] = xv.v[c];
  }
  if (conv_ok) {
#pragma unroll
    for (int q = 0; q < S; ++q)
      st_stream(reinterpret_cast<V8*>(st) + q, *reinterpret_cast<const V8*>(&ns.v[8 * q]));
  }
}

template <int K, int V, typename T, typename GT, typename BT>
__global__ void __launch_bounds__(kFusedThreads) gdn_conv_decode_kernel(FusedParams p) {
  constexpr int NT = kFusedThreads;
  __shared__ __align__(16) Partials<V, NT> red;
  __shared__ __align__(16) float xv_lds[K * 2];  // q and k after conv + SiLU
  __shared__ __align__(16) float vv_lds[16][V];          // v heads of the group (R <= 16)
  const int64_t b = blockIdx.x / p.H;
  const int h = static_cast<int>(blockIdx.x % p.H);
  const int R = p.HV / p.H;
  const int tid = threadIdx.x;
  const int64_t cslot = p.conv_idx ? p.conv_idx[b] : b;
  const int64_t sslot = p.ssm_idx ? p.ssm_idx[b] : b;
  if (p.conv_idx && cslot == p.pad) return;  // padded batch row

  // Conv update for the group's channels: q (K), k (K), then R * V of v.
  const int nch = 2 * K + R * V;
  const bool conv_ok = cslot >= 0 && cslot < p.conv_lines;
  const bool st_ok = sslot >= 0 && sslot < p.slots;
  // The first v head's state tile is requested before the conv phase, so
  // its 64 KB stream overlaps the conv loads and arithmetic.
  Tile<K, V, NT> t;
  {
    float* sbase = p.state + sslot * p.st_slot_stride + static_cast<int64_t>(h) * R * K * V;
    if (st_ok) load_tile<K, V>(t, sbase); else zero_tile<K, V>(t);
  }
  // Global channel of group channel i: q (K), k (K), then R * V of v.
  auto chan = [&](int i) -> int64_t {
    if (i < K) return static_cast<int64_t>(h) * K + i;
    if (i < 2 * K) return static_cast<int64_t>(p.H) * K + static_cast<int64_t>(h) * K + (i - K);
    return 2 * static_cast<int64_t>(p.H) * K + static_cast<int64_t>(h) * R * V + (i - 2 * K);
  };
  auto put = [&](int i, float y) {
    if (i < 2 * K) xv_lds[i] = y;
    else vv_lds[(i - 2 * K) / V][(i - 2 * K) % V] = y;
  };
  if (p.conv_vec) {
    // 8 channels per lane (K and V are multiples of 8, so a group never
    // straddles the q / k / v parts).
    for (int i = tid * 8; i < nch; i += NT * 8) {
      float y[8];
      switch (p.S) {
        case 1: conv8<T, 1>(p, b, cslot, conv_ok, chan(i), y); break;
        case 2: conv8<T, 2>(p, b, cslot, conv_ok, chan(i), y); break;
        case 3: conv8<T, 3>(p, b, cslot, conv_ok, chan(i), y); break;
        default: conv8<T, 4>(p, b, cslot, conv_ok, chan(i), y); break;
      }
#pragma unroll
      for (int c = 0; c < 8; ++c) put(i + c, y[c]);
    }
  } else {
  for (int i = tid; i < nch; i += NT) {
    int64_t ch;
    if (i < K) ch = static_cast<int64_t>(h) * K + i;
    else if (i < 2 * K) ch = static_cast<int64_t>(p.H) * K + static_cast<int64_t>(h) * K + (i - K);
    else ch = 2 * static_cast<int64_t>(p.H) * K + static_cast<int64_t>(h) * R * V + (i - 2 * K);
    const float xc = ldf<T>(p.x, b * p.sx + ch);
    float acc = p.cbias ? load_as_f32(p.cbias, ch, p.wdt) : 0.f;
    T* st = reinterpret_cast<T*>(p.conv_state) + cslot * p.cs_line + ch * p.cs_dim;
    // window = cat(state[S-W+1 .. S-1], x)
    for (int j = 0; j < p.W - 1; ++j) {
      const float sv = conv_ok ? to_f32(st[(p.S - p.W + 1 + j) * p.cs_tok]) : 0.f;
      acc = fmaf(sv, load_as_f32(p.w, ch * p.w_dim + j * p.w_tap, p.wdt), acc);
    }
    acc = fmaf(xc, load_as_f32(p.w, ch * p.w_dim + (p.W - 1) * p.w_tap, p.wdt), acc);
    const float y = silu(acc);
    if (conv_ok) {  // shift the state left by one and append x
      for (int j = 0; j + 1 < p.S; ++j) st[j * p.cs_tok] = st[(j + 1) * p.cs_tok];
      st[(p.S - 1) * p.cs_tok] = reinterpret_cast<const T*>(p.x)[b * p.sx + ch];
    }
    put(i, y);
  }
  }
  __syncthreads();

  // Head j's tile is in `cur`; the next head's tile streams into `nxt`
  // while head j computes (two register tiles, unrolled by two): 204.4 ->
  // 197.8 us at config 5 on MI355X, the state stream no longer pausing
  // between the group's heads.
  const QkScales sc = qk_scales<K>(xv_lds, xv_lds + K, p.l2norm, p.scale);
  Tile<K, V, NT> t2;
  auto head = [&](Tile<K, V, NT>& cur, Tile<K, V, NT>& nxt, int j) {
    const int hv = h * R + j;
    float* sbase = p.state + sslot * p.st_slot_stride + static_cast<int64_t>(hv) * K * V;
    if (j + 1 < R) {
      if (st_ok) load_tile<K, V>(nxt, sbase + K * V); else zero_tile<K, V>(nxt);
    }
    float gv = ldf<GT>(p.g, b * p.HV + hv);
    float beta = p.beta ? ldf<BT>(p.beta, b * p.HV + hv) : 1.0f;
    if (p.gating) {
      gv = gdn_log_decay(gv + p.dt_bias[hv], p.A_log[hv], p.sp_beta, 1.0f / p.sp_beta, p.sp_thr);
      beta = sigmoid_exact(beta);
    }
    T* o = reinterpret_cast<T*>(p.o) + (b * p.HV + hv) * V;
    gdn_token<K, V>(
        cur, red, j & 1, xv_lds, xv_lds + K, vv_lds[j], sc, __expf(gv), beta, [] {},
        [&](int c, const float (&val)[4]) {
#pragma unroll
          for (int u = 0; u < 4; ++u) o[c + u] = from_f32<T>(val[u]);
        });
    if (st_ok) store_tile<K, V>(cur, sbase);
  };
  for (int j = 0; j < R; j += 2) {
    head(t, t2, j);
    if (j + 1 < R) head(t2, t, j + 1);
  }
}

template <int K, int V, typename T, typename GT>
int fused_beta(const FusedParams& p, xk_dtype bdt, hipStream_t s) {
  const dim3 grid(p.B * p.H);
  switch (bdt) {
    case XK_F32: hipLaunchKernelGGL((gdn_conv_decode_kernel<K, V, T, GT, float>), grid, dim3(kFusedThreads), 0, s, p); break;
    case XK_BF16: hipLaunchKernelGGL((gdn_conv_decode_kernel<K, V, T, GT, bf16>), grid, dim3(kFusedThreads), 0, s, p); break;
    case XK_F16: hipLaunchKernelGGL((gdn_conv_decode_kernel<K, V, T, GT, f16>), grid, dim3(kFusedThreads), 0, s, p); break;
    default: return XK_ERR_UNSUPPORTED;
  }
  return launch_status();
}

template <int K, int V, typename T>
int fused_g(const FusedParams& p, xk_dtype gdt, xk_dtype bdt, hipStream_t s) {
  switch (gdt) {
    case XK_F32: return fused_beta<K, V, T, float>(p, bdt, s);
    case XK_BF16: return fused_beta<K, V, T, bf16>(p, bdt, s);
    case XK_F16: return fused_beta<K, V, T, f16>(p, bdt, s);
    default: return XK_ERR_UNSUPPORTED;
  }
}

}  // namespace
}  // namespace xk

using namespace xk;

extern "C" int xk_gdn_recurrent_strided(
    const void* q, int64_t stride_q_tok, const void* k, int64_t stride_k_tok, const void* v,
    int64_t stride_v_tok, xk_dtype dtype, const void* g,
    xk_dtype g_dtype, const void* beta, xk_dtype beta_dtype, void* o,
    const float* initial_state, int64_t stride_h0_slot, float* final_state,
    int64_t stride_ht_slot, int64_t num_slots, const void* cu_seqlens,
    xk_dtype cu_dtype, const int32_t* ssm_state_indices, int64_t stride_idx_seq,
    int64_t stride_idx_tok, const int32_t* num_accepted_tokens, int64_t N,
    int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V, float scale,
    int use_qk_l2norm, int inplace_final_state, void* stream) {
  if (N < 0 || T < 0 || H <= 0 || HV <= 0 || HV % H != 0) return XK_ERR_INVALID;
  if (stride_q_tok < H * K || stride_k_tok < H * K || stride_v_tok < HV * V) return XK_ERR_INVALID;
  if (!is_float_dtype(dtype) || !is_float_dtype(g_dtype) ||
      (beta && !is_float_dtype(beta_dtype)))
    return XK_ERR_UNSUPPORTED;
  if (cu_seqlens && cu_dtype != XK_I32 && cu_dtype != XK_I64) return XK_ERR_UNSUPPORTED;
  if (N == 0) return XK_OK;
  if (!q || !k || !v || !g || !o || !final_state) return XK_ERR_INVALID;
  if (inplace_final_state && !ssm_state_indices) return XK_ERR_INVALID;
  if (num_accepted_tokens && (!ssm_state_indices || !cu_seqlens || stride_idx_tok == 0))
    return XK_ERR_INVALID;
  if (!aligned(initial_state, 16) || !aligned(final_state, 16) ||
      stride_h0_slot % 4 || stride_ht_slot % 4)
    return XK_ERR_INVALID;
  RecParams p{};
  p.q = q;
  p.k = k;
  p.v = v;
  p.sq = stride_q_tok;
  p.sk = stride_k_tok;
  p.sv = stride_v_tok;
  p.g = g;
  p.beta = beta;
  p.o = o;
  p.h0 = initial_state;
  p.ht = final_state;
  p.h0_slot_stride = stride_h0_slot;
  p.ht_slot_stride = stride_ht_slot;
  p.slots = num_slots;
  p.cu = cu_seqlens;
  p.cu_i64 = cu_dtype == XK_I64;
  p.idx = ssm_state_indices;
  p.idx_s0 = stride_idx_seq;
  p.idx_s1 = stride_idx_tok;
  p.accepted = num_accepted_tokens;
  p.N = N;
  p.T = T;
  p.H = static_cast<int>(H);
  p.HV = static_cast<int>(HV);
  p.scale = scale;
  p.l2norm = use_qk_l2norm;
  p.inplace = inplace_final_state;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const xk_dtype bdt = beta ? beta_dtype : XK_F32;
  if (K == 128 && V == 128) return rec_t<128, 128>(p, dtype, g_dtype, bdt, s);
  if (K == 64 && V == 64) return rec_t<64, 64>(p, dtype, g_dtype, bdt, s);
  if (K == 128 && V == 64) return rec_t<128, 64>(p, dtype, g_dtype, bdt, s);
  if (K == 64 && V == 128) return rec_t<64, 128>(p, dtype, g_dtype, bdt, s);
  return XK_ERR_UNSUPPORTED;
}

extern "C" int xk_gdn_recurrent(
    const void* q, const void* k, const void* v, xk_dtype dtype, const void* g,
    xk_dtype g_dtype, const void* beta, xk_dtype beta_dtype, void* o,
    const float* initial_state, int64_t stride_h0_slot, float* final_state,
    int64_t stride_ht_slot, int64_t num_slots, const void* cu_seqlens,
    xk_dtype cu_dtype, const int32_t* ssm_state_indices, int64_t stride_idx_seq,
    int64_t stride_idx_tok, const int32_t* num_accepted_tokens, int64_t N,
    int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V, float scale,
    int use_qk_l2norm, int inplace_final_state, void* stream) {
  return xk_gdn_recurrent_strided(q, H * K, k, H * K, v, HV * V, dtype, g, g_dtype, beta,
                                  beta_dtype, o, initial_state, stride_h0_slot, final_state,
                                  stride_ht_slot, num_slots, cu_seqlens, cu_dtype,
                                  ssm_state_indices, stride_idx_seq, stride_idx_tok,
                                  num_accepted_tokens, N, T, H, HV, K, V, scale, use_qk_l2norm,
                                  inplace_final_state, stream);
}

namespace {

// Shared argument checks and launch of the fused decode step; p.g / p.beta
// (and, with p.gating, a / b) are already set.
int conv_decode_launch(FusedParams& p, const void* mixed_qkv, int64_t stride_x_row,
                       void* conv_state, int64_t stride_cs_line, int64_t stride_cs_dim,
                       int64_t stride_cs_tok, int64_t conv_lines, int64_t conv_state_len,
                       const void* conv_weight, int64_t stride_w_dim, int64_t stride_w_tap,
                       const void* conv_bias, xk_dtype w_dtype, int64_t width,
                       const int32_t* conv_state_indices, int32_t pad_slot_id, xk_dtype g_dtype,
                       xk_dtype beta_dtype, float* ssm_state, int64_t stride_state_slot,
                       int64_t num_slots, const int32_t* ssm_state_indices, void* o, int64_t B,
                       int64_t H, int64_t HV, int64_t K, int64_t V, float scale,
                       int use_qk_l2norm, xk_dtype dtype, void* stream) {
  if (B < 0 || H <= 0 || HV <= 0 || HV % H != 0 || HV / H > 16 || width < 1 ||
      conv_state_len < width - 1 || conv_state_len < 1)
    return XK_ERR_INVALID;
  if (!is_float_dtype(dtype) || !is_float_dtype(g_dtype) || !is_float_dtype(w_dtype) ||
      (p.beta && !is_float_dtype(beta_dtype)))
    return XK_ERR_UNSUPPORTED;
  if (B == 0) return XK_OK;
  if (!mixed_qkv || !conv_state || !conv_weight || !p.g || !ssm_state || !o)
    return XK_ERR_INVALID;
  if (!aligned(ssm_state, 16) || stride_state_slot % 4) return XK_ERR_INVALID;
  if (K != 128 || V != 128) return XK_ERR_UNSUPPORTED;
  p.x = mixed_qkv;
  p.sx = stride_x_row;
  p.conv_state = conv_state;
  p.cs_line = stride_cs_line;
  p.cs_dim = stride_cs_dim;
  p.cs_tok = stride_cs_tok;
  p.conv_lines = conv_lines;
  p.S = static_cast<int>(conv_state_len);
  p.w = conv_weight;
  p.w_dim = stride_w_dim;
  p.w_tap = stride_w_tap;
  p.cbias = conv_bias;
  p.wdt = w_dtype;
  p.conv_idx = conv_state_indices;
  p.W = static_cast<int>(width);
  p.state = ssm_state;
  p.st_slot_stride = stride_state_slot;
  p.slots = num_slots;
  p.ssm_idx = ssm_state_indices;
  p.o = o;
  p.B = B;
  p.H = static_cast<int>(H);
  p.HV = static_cast<int>(HV);
  p.scale = scale;
  p.l2norm = use_qk_l2norm;
  p.pad = pad_slot_id;
  p.conv_vec = (dtype == XK_BF16 || dtype == XK_F16) && w_dtype == dtype &&
               stride_w_dim == width && stride_w_tap == 1 && stride_cs_tok == 1 &&
               stride_cs_dim == conv_state_len && conv_state_len == width - 1 &&
               conv_state_len <= 4 && stride_cs_line % 8 == 0 && stride_x_row % 8 == 0 &&
               aligned(mixed_qkv, 16) && aligned(conv_state, 16) && aligned(conv_weight, 16);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const xk_dtype bdt = p.beta ? beta_dtype : XK_F32;
  switch (dtype) {
    case XK_BF16: return fused_g<128, 128, bf16>(p, g_dtype, bdt, s);
    case XK_F16: return fused_g<128, 128, f16>(p, g_dtype, bdt, s);
    case XK_F32: return fused_g<128, 128, float>(p, g_dtype, bdt, s);
    default: return XK_ERR_UNSUPPORTED;
  }
}

}  // namespace

extern "C" int xk_gdn_conv_decode(
    const void* mixed_qkv, int64_t stride_x_row, void* conv_state,
    int64_t stride_cs_line, int64_t stride_cs_dim, int64_t stride_cs_tok,
    int64_t conv_lines, int64_t conv_state_len, const void* conv_weight,
    int64_t stride_w_dim, int64_t stride_w_tap, const void* conv_bias,
    xk_dtype w_dtype, int64_t width, const int32_t* conv_state_indices,
    int32_t pad_slot_id, const void* g, xk_dtype g_dtype, const void* beta,
    xk_dtype beta_dtype, float* ssm_state, int64_t stride_state_slot,
    int64_t num_slots, const int32_t* ssm_state_indices, void* o, int64_t B,
    int64_t H, int64_t HV, int64_t K, int64_t V, float scale,
    int use_qk_l2norm, xk_dtype dtype, void* stream) {
  FusedParams p{};
  p.g = g;
  p.beta = beta;
  return conv_decode_launch(p, mixed_qkv, stride_x_row, conv_state, stride_cs_line,
                            stride_cs_dim, stride_cs_tok, conv_lines, conv_state_len,
                            conv_weight, stride_w_dim, stride_w_tap, conv_bias, w_dtype, width,
                            conv_state_indices, pad_slot_id, g_dtype, beta_dtype, ssm_state,
                            stride_state_slot, num_slots, ssm_state_indices, o, B, H, HV, K, V,
                            scale, use_qk_l2norm, dtype, stream);
}

extern "C" int xk_gdn_conv_gating_decode(
    const void* mixed_qkv, int64_t stride_x_row, void* conv_state,
    int64_t stride_cs_line, int64_t stride_cs_dim, int64_t stride_cs_tok,
    int64_t conv_lines, int64_t conv_state_len, const void* conv_weight,
    int64_t stride_w_dim, int64_t stride_w_tap, const void* conv_bias,
    xk_dtype w_dtype, int64_t width, const int32_t* conv_state_indices,
    int32_t pad_slot_id, const float* A_log, const void* a, const float* dt_bias,
    const void* b, xk_dtype ab_dtype, float softplus_beta, float threshold,
    float* ssm_state, int64_t stride_state_slot, int64_t num_slots,
    const int32_t* ssm_state_indices, void* o, int64_t B, int64_t H, int64_t HV,
    int64_t K, int64_t V, float scale, int use_qk_l2norm, xk_dtype dtype,
    void* stream) {
  if (B > 0 && (!A_log || !dt_bias || !a || !b)) return XK_ERR_INVALID;
  if (softplus_beta == 0.f) return XK_ERR_INVALID;
  FusedParams p{};
  p.g = a;
  p.beta = b;
  p.gating = 1;
  p.A_log = A_log;
  p.dt_bias = dt_bias;
  p.sp_beta = softplus_beta;
  p.sp_thr = threshold;
  return conv_decode_launch(p, mixed_qkv, stride_x_row, conv_state, stride_cs_line,
                            stride_cs_dim, stride_cs_tok, conv_lines, conv_state_len,
                            conv_weight, stride_w_dim, stride_w_tap, conv_bias, w_dtype, width,
                            conv_state_indices, pad_slot_id, ab_dtype, ab_dtype, ssm_state,
                            stride_state_slot, num_slots, ssm_state_indices, o, B, H, HV, K, V,
                            scale, use_qk_l2norm, dtype, stream);
}

extern "C" int xk_fused_gdn_gating(const float* A_log, const void* a, const void* b,
                                   const float* dt_bias, float* g_out, void* beta_out,
                                   int64_t rows, int64_t heads, float softplus_beta,
                                   float threshold, xk_dtype ab_dtype, void* stream) {
  if (rows < 0 || heads <= 0 || heads > INT32_MAX || softplus_beta == 0.f) return XK_ERR_INVALID;
  if (!is_float_dtype(ab_dtype)) return XK_ERR_UNSUPPORTED;
  if (rows == 0) return XK_OK;
  if (!A_log || !a || !b || !dt_bias || !g_out || !beta_out) return XK_ERR_INVALID;
  const int64_t n = rows * heads;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int hh = static_cast<int>(heads);
#define XK_GATE(T, IT)                                                                       \
  hipLaunchKernelGGL((gdn_gating_kernel<T, IT>), dim3(cdiv(n, kGateBlock)), dim3(kGateBlock), 0, \
                     s, A_log,                                                                 \
                     static_cast<const T*>(a), static_cast<const T*>(b), dt_bias, g_out,        \
                     static_cast<T*>(beta_out), static_cast<IT>(n), hh, softplus_beta,          \
                     1.0f / softplus_beta, threshold)
#define XK_GATE_T(T)                                   \
  if (n + kGateBlock < (int64_t{1} << 31)) {           \
    XK_GATE(T, uint32_t);                              \
  } else {                                             \
    XK_GATE(T, int64_t);                               \
  }
  switch (ab_dtype) {
    case XK_BF16: XK_GATE_T(bf16); break;
    case XK_F16: XK_GATE_T(f16); break;
    default: XK_GATE_T(float); break;
  }
#undef XK_GATE_T
#undef XK_GATE
  return launch_status();
}

extern "C" int xk_gdn_sigmoid_gating_update(
    const float* A_log, const void* a, const float* dt_bias, float softplus_beta,
    float threshold, const void* q, const void* k, const void* v, const void* b,
    xk_dtype ab_dtype, void* o, float* state, int64_t stride_state_slot,
    int64_t num_slots, const int32_t* state_indices, const int32_t* cu_seqlens,
    int64_t N, int64_t H, int64_t HV, int64_t K, int64_t V, float scale,
    int use_qk_l2norm, xk_dtype dtype, void* stream) {
  if (N < 0 || H <= 0 || HV <= 0 || HV % H != 0 || softplus_beta == 0.f) return XK_ERR_INVALID;
  if (!is_float_dtype(dtype) || !is_float_dtype(ab_dtype)) return XK_ERR_UNSUPPORTED;
  if (N == 0) return XK_OK;
  if (!A_log || !a || !dt_bias || !q || !k || !v || !b || !o || !state || !state_indices ||
      !cu_seqlens)
    return XK_ERR_INVALID;
  if (!aligned(state, 16) || stride_state_slot % 4) return XK_ERR_INVALID;
  RecParams p{};
  p.q = q;
  p.k = k;
  p.v = v;
  p.sq = p.sk = H * K;
  p.sv = HV * V;
  p.g = a;
  p.beta = b;
  p.o = o;
  p.h0 = state;
  p.ht = state;
  p.h0_slot_stride = stride_state_slot;
  p.ht_slot_stride = stride_state_slot;
  p.slots = num_slots;
  p.cu = cu_seqlens;
  p.cu_i64 = 0;
  p.idx = state_indices;
  p.idx_s0 = 1;
  p.idx_s1 = 0;
  p.accepted = nullptr;
  p.N = N;
  p.T = 0;
  p.H = static_cast<int>(H);
  p.HV = static_cast<int>(HV);
  p.scale = scale;
  p.l2norm = use_qk_l2norm;
  p.inplace = 1;
  p.gating = 1;
  p.A_log = A_log;
  p.dt_bias = dt_bias;
  p.sp_beta = softplus_beta;
  p.sp_thr = threshold;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (K == 128 && V == 128) return rec_t<128, 128>(p, dtype, ab_dtype, ab_dtype, s);
  if (K == 64 && V == 64) return rec_t<64, 64>(p, dtype, ab_dtype, ab_dtype, s);
  if (K == 128 && V == 64) return rec_t<128, 64>(p, dtype, ab_dtype, ab_dtype, s);
  if (K == 64 && V == 128) return rec_t<64, 128>(p, dtype, ab_dtype, ab_dtype, s);
  return XK_ERR_UNSUPPORTED;
}
