// Chunked gated delta rule (prefill) for gfx950, chunk size 64.
//
// Semantics follow chunk_gated_delta_rule_full_op_ref
// (triton_npu/test/triton_chunk_gated_delta_rule_test.cpp:190-323), the
// pipeline of triton_npu/triton_src/chunk_gated_delta_rule/chunk.py:32-80.
// Per sequence, per v-head, per 64-token chunk with in-chunk cumulative
// log-decay gc (cumsum.py), beta b, keys k, queries q (scaled), values v and
// carried state S [K, V] (fp32):
//   M    = strict_tril(b_i (k_i . k_j) exp(gc_i - gc_j))     (kkt.py)
//   Ai   = (I + M)^-1                                        (solve_tril.py)
//   Vn   = Ai (b * (v - exp(gc) * (k S)))     == u - w S      (wy_fast.py,
//                                                            chunk_delta_h.py)
//   o    = exp(gc) * (q S) + tril(q k^T * exp(gc_i - gc_j)) Vn (chunk_o.py)
//   S   <- exp(gc_last) S + k^T (exp(gc_last - gc) * Vn)
// GQA: v-head hv uses qk-head hv / (HV / H).  Optional l2norm of q and k
// (npu_l2norm_last_dim, x / sqrt(sum x^2 + 1e-6)) is folded in as per-token
// row scales, so the matrix products always see the exact bf16 inputs.
//
// Two launches (three above 64 sequences, four with segments), no host
// synchronisation (capturable in a hipGraph):
//  * P0 (one small block, above 64 sequences) turns cu_seqlens into chunk
//    offsets.
//  * P1, fully parallel, one wave per (chunk, v-head), computes everything
//    that does not depend on the carried state and writes one record per
//    (chunk, head) to the workspace:
//      - Ai = (I + M)^-1 as a bf16 hi/lo pair (hi + lo carries ~16 mantissa
//        bits).  K K^T runs on bf16 MFMA (exact products, fp32 sums); the
//        inverse inverts the four 16x16 diagonal blocks by forward
//        substitution (one lane per column) and merges them, X10 = -X11 M10
//        X00, with hi/lo-split MFMAs (invert_unit_lower);
//      - Aq = scale * tril(r_q r_k (q k^T) exp(gc_i - gc_j)) in bf16 (it only
//        feeds the bf16 output);
//      - per-token factors cq = scale exp(gc) r_q, ck = b exp(gc) r_k, b,
//        ed = r_k exp(gc_last - gc), and exp(gc_last).
//  * P2, sequential over the chunks of a sequence, one 512-lane block per
//    (sequence, v-head, 64-column V tile) (gdn_chunk_state8_kernel; a
//    256-lane block per 32-column tile when V is not a multiple of 64),
//    carries the fp32 state tile in registers through the short dependent
//    chain
//      KS = K S -> R = b v - ck KS -> Vn = Ai R -> S = e^gl S + K^T (ed Vn)
//    (hi/lo-split bf16 MFMAs keep the state within fp32-reference tolerance)
//    and emits o = cq (Q S) + Aq Vn.  Every global operand of chunk c+1 is
//    loaded while chunk c computes.  Blocks of one (sequence, head) share an
//    XCD (block id mod 8) and thus its L2 for the shared q/k/record reads.
//    Where few blocks would leave the chip idle behind long sequences, P2
//    runs as three passes over segments of them ("Segments" below).
#include <algorithm>
#include <atomic>
#include <mutex>

#include "gdn_common.h"

namespace xk {
namespace {

using namespace gdn;

constexpr int kBVMax = 64;  // most V columns per P2 block (32 or 64)
constexpr int kTh = 256;  // threads per block
// Per-(chunk, head) record: ai_hi, ai_lo, aq, then the per-token factors
// (fp32 [5][64]: cq, ck, b, ed, exp(gc_last)).  Each matrix is stored as the
// MFMA A-operand images the state kernel loads, 1 KB each with lane l's 16
// bytes at byte 16 l: image (w, kk) holds rows 16 w + l % 16, columns
// 32 kk + 8 (l / 16) .. + 7, for wave w's rows.  The matrices are lower
// triangular, so the zero upper-right 32 x 32 block has no image: waves 0
// and 1 (rows 0..31) have only kk = 0, six images in all.  A lane-per-row
// layout (each load instruction touching 16 rows, 64 bytes of each) made
// the state kernel 15 us slower (262 -> 277 us at config 4 on MI355X): the
// loads of adjacent lanes were not contiguous.
constexpr int kMat = 6 * 512 * 2;  // bf16 bytes per matrix
constexpr int kRec = 3 * kMat + 5 * kC * 4;    // 19712 = 77 * 256
static_assert(kRec % 256 == 0, "records stay 256-byte aligned");

// Image of operand kk of wave w (waves 0, 1: kk = 0 only; their kk = 1
// maps to the kk = 0 image).
__device__ __forceinline__ int img_index(int w, int kk) { return w < 2 ? w : 2 * w - 2 + kk; }
// Padded rows of a sequence's last chunk store their (unused) outputs here,
// so that every store in the chunk loop is unconditional: gfx9 counts loads
// and stores in one in-order counter, and a store that only some paths
// issue makes the compiler wait for every outstanding prefetch.
constexpr int kDump = kC * kBVMax * 2;

struct ChunkParams {
  const void* q;  // [T, H, K], token pitch sqk
  const void* k;
  const void* v;  // [T, HV, V], token pitch sv
  uint32_t sqk, sv;  // elements; views of a wider row (the conv's output) are read in place
  const void* g;  // [T, HV]
  const void* beta;
  void* o;  // [T, HV, V]
  const float* h0;  // [N, HV, K, V] or NULL
  float* ht;        // [N, HV, K, V] or NULL
  const void* cu;   // [N+1]
  int cu_i64;
  int32_t* chunk_off;  // [N+1] workspace
  int32_t* seq_order;  // [N] workspace: sequences, longest first
  int2* ctab;          // [NTmax] workspace: (first token, length) per chunk
  // [N], N <= kWaveSeqs, in the place of the three above (which are unused
  // then): sequence, first global chunk, first and end token of rank r,
  // longest first.
  int4* seqtab;
  bf16* dump;          // [64 * kBVMax] workspace: sink for padded-row stores
  char* rec;           // [NTmax, HV] records of kRec bytes, workspace
  int64_t N, NTmax;
  int64_t T;  // token rows of q/k/v
  int H, HV;
  float scale;
  int l2norm;
  // Segmented state pass (below); seg_max 0: whole sequences only.
  int seg_max;        // segments the workspace holds
  int seg_cus, seg_nvt;  // compute units and V tiles the plan counts on
  int32_t* seg_len;   // the plan: chunks per segment
  char* seg_m;        // [seg_max, HV]: transition M - c I of a segment, kSegImg bytes of operand images
  float* seg_c;       // [seg_max, HV]: c, the product of the segment's decays
  float* seg_b;       // [seg_max, HV, K, V]: its end state from zero (the first one's: from h0),
                      // then the state after it
  int32_t* seg_over;  // [seg_max, HV, 2]: an entry of that half of M - c I, or c, exceeds kSegLimit
  int32_t* seg_bad;   // [N, HV]: the head runs in order
};

__device__ __forceinline__ char* rec_at(const ChunkParams& p, int64_t c, int hv) {
  return p.rec + (c * p.HV + hv) * static_cast<int64_t>(kRec);
}

// ---------------------------------------------------------------------------
// Segments.  A sequence's chunk chain is serial, so few (sequence, head, V
// tile) blocks leave most CUs idle behind a long chain.  A sequence may be
// cut into segments of `len` chunks that run in parallel:
//  * kSegSum: per segment, the state after it from a zero state (B; the
//    first segment starts from the initial state instead) and its transition
//    M (the same recurrence without values, from the identity: K more
//    columns), without outputs;
//  * gdn_chunk_combine_kernel: the states at the segment boundaries,
//    S <- M_i S + B_i in order, as c_i S + (M_i - c_i I) S + B_i with c_i the
//    product of the segment's decays, to fp32 precision;
//  * kSegOut: every segment from its entry state, with outputs.
// The work of the state pass grows about 2.4 times, so this pays only where
// the chip is idle.  len is chosen on the device, where the lengths are
// known: one block of the prep kernel evaluates seg_cost for 1 .. 64
// segments of the longest sequence, one candidate per lane.  The host
// launches these passes if a batch of this size gains whatever its lengths
// (seg_plan).  MI355X, us per call of the whole op without and with segments:
// one sequence of 8 v-heads, 1,024 tokens 52 and 50, 4,096 tokens 175 and 77,
// 32,768 tokens 1266 and 280; 2 sequences of 4,096 x 16 v-heads 180 and 140.
//
// A chunk of the chain in order scales the state in fp32 and rounds only what
// the delta rule adds (bf16 hi/lo operands).  A boundary must lose no more:
// M in hi/lo images would round the whole state to 2^-17 there however little
// the segment changes it (final states of heads with beta ~ 0.01 and decays
// ~ 1e-5 a token were 15 to 30 times as far from 64 bits as in order).  With
// c split off and 24-bit products the errors of the two are the same.
//
// An entry of M - c I (or c) outside [-kSegLimit, kSegLimit] (or NaN) makes
// the whole head run in order: with keys of norm <= 1, beta in [0, 1] and
// decays <= 1 a transition has norm <= 1; without these its products could
// overflow or cancel where the chain in order does not.
// ---------------------------------------------------------------------------
constexpr float kSegLimit = 2.f;
constexpr int64_t kSegImg = 128 * 128 * 6;  // three bf16 images of one transition's operands
constexpr int64_t kSegSeqs = 16;            // most sequences (the plan loops over them)

// Time of the state pass (us) when the longest sequence is cut into `s`
// segments of `len` chunks: `sums` kSegSum blocks and `outs` kSegOut blocks in
// rounds of one per CU.  `sums` includes the transition blocks of first
// segments, which end at once: an XCD hands its blocks to its shader engines
// in turn, and with four tiles per (segment, head) all of one kind fall to
// one engine, so the places that idle blocks leave are not taken by others
// (3 segments x 24 heads, 240 blocks of 288 with work, take two rounds of 256
// CUs).  A step takes 1.6 (sum) or 2.35 us (out) on an idle chip and about
// 0.6 us more on one full of blocks with work (`work` of the sums; idle ones
// counted there kept 2 sequences of 8,689 tokens x 32 v-heads whole, 432 us
// against 411), a step of the combine kernel 1.4 us.  Against
// traced passes (MI355X, one sequence of 8 v-heads) the sum of the three is
// 68 (model) and 66 us at 4,096 tokens (8 segments), 277 and 260 at 32,768
// (16).
__host__ __device__ inline float seg_cost(int s, int len, int sums, int work, int outs,
                                          int cus) {
  auto time = [&](int blocks, int busy, float step) {
    const float load = static_cast<float>(busy) / cus;
    return fmaxf(1.f, ceilf(static_cast<float>(blocks) / cus)) * len * (step + 0.6f * fminf(1.f, load));
  };
  const float out = 8.f + time(outs, outs, 2.35f);
  return s <= 1 ? out : out + 14.f + time(sums, work, 1.6f) + 1.4f * (s - 2);
}

// Chunks per segment for this batch, 0 for whole sequences (wave-uniform; N <=
// kSegSeqs).
__device__ __forceinline__ int wave_seg_len(const ChunkParams& p) {
  const int lane = threadIdx.x & (kWave - 1);
  const int N = static_cast<int>(p.N);
  const WaveSeqs w = wave_seqs(p);
  int longest = 1;
  for (int n = 0; n < N; ++n) longest = max(longest, __builtin_amdgcn_readlane(w.cnt, n));
  const int len = (longest + lane) / (lane + 1);
  int segs = 0, cut = 0;  // cut: sequences of several segments
  for (int n = 0; n < N; ++n) {
    const int c = (__builtin_amdgcn_readlane(w.cnt, n) + len - 1) / len;
    segs += max(c, 1);
    cut += c > 1;
  }
  const int sums = (segs - N) * (p.seg_nvt + 2) * p.HV;
  const float cost = seg_cost(lane + 1, len, sums, sums - cut * 2 * p.HV,
                              segs * p.seg_nvt * p.HV, p.seg_cus);
  // Smallest cost, the fewest segments among equals.
  int key = lane == 0 || segs <= p.seg_max ? static_cast<int>(fminf(cost * 16.f, 3e7f)) : 30000000;
  key = key * kWave + lane;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) key = min(key, __shfl_xor(key, o, kWave));
  const int best = __builtin_amdgcn_readfirstlane(key & (kWave - 1));
  return best ? __builtin_amdgcn_readlane(len, best) : 0;
}

struct WaveSegs {
  WaveSeqs s;
  int len;       // chunks per segment, 0: whole sequences
  int32_t cnt;   // sequence lane's segments (an empty sequence has one)
  int32_t incl;  // segments of sequences 0 .. lane
};
__device__ __forceinline__ WaveSegs wave_segs(const ChunkParams& p) {
  WaveSegs w;
  w.len = *p.seg_len;
  w.s = wave_seqs(p);
  const int lane = threadIdx.x & (kWave - 1);
  w.cnt = lane >= p.N ? 0 : w.len ? max((w.s.cnt + w.len - 1) / w.len, 1) : 1;
  w.incl = wave_incl_scan(w.cnt);
  return w;
}

// Sequence of rank r (wave-uniform).
struct SeqEntry {
  int64_t n, c0, bos, eos;
};
__device__ __forceinline__ SeqEntry ranked_seq(const ChunkParams& p, int64_t r) {
  if (p.N <= kWaveSeqs) {
    const int4 e = p.seqtab[r];
    return {e.x, e.y, e.z, e.w};
  }
  const int64_t n = p.seq_order[r];
  return {n, p.chunk_off[n], cu_at(p, n), cu_at(p, n + 1)};
}

// Rows >= L of the K / Q operands (q4_load) repeat row L-1; here every
// consumer zeroes them through factors that are 0 there (beta, ck, ed, the
// masks of M and Aq).

// ---------------------------------------------------------------------------
// P1: one wave per (chunk, v-head); waves of a block are independent.
// ---------------------------------------------------------------------------

// r[row] = 1 / sqrt(sum x^2 + 1e-6) for the 64 rows of a chunk held as MFMA
// A operands (lane: row mi*16 + l15, elements kk*32 + 8*lg ...), or 1 when
// `on` is 0.  Sums use bf16 dot2 (exact products, fp32 accumulation).
template <int KK>
__device__ __forceinline__ void row_scales(const bf8_t (&x)[4][KK], float* r, int on) {
  const int lane = threadIdx.x & 63;
  const int l15 = lane & 15, lg = lane >> 4;
  if (!on) {
    if (lg == 0)
#pragma unroll
      for (int mi = 0; mi < 4; ++mi) r[mi * 16 + l15] = 1.0f;
    return;
  }
#pragma unroll
  for (int mi = 0; mi < 4; ++mi) {
    float ss = 0.f;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const bf2_t pr = {x[mi][kk][e], x[mi][kk][e + 1]};
        ss = __builtin_amdgcn_fdot2_f32_bf16(pr, pr, ss, false);
      }
    ss += __shfl_xor(ss, 16, kWave);
    ss += __shfl_xor(ss, 32, kWave);
    if (lg == 0) r[mi * 16 + l15] = 1.0f / sqrtf(ss + 1e-6f);
  }
}

template <int K, typename GT, typename BT>
__global__ void __launch_bounds__(kTh) gdn_chunk_prep_kernel(ChunkParams p) {
  __shared__ __align__(16) float lds[4][kC][kLd];
  __shared__ __align__(16) float vec[4][5][kC];  // gc, beta, r_k, r_q, c_k per wave
  // Wave index in a scalar register: the exit below is then a scalar branch,
  // and the DPP transposes (q4_to_a) run with every lane of the wave active.
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int l15 = lane & 15, lg = lane >> 4;
  // Blocks take the head groups of one chunk before the next chunk, so
  // that the blocks in flight read whole token rows.
  const int hg4 = (p.HV + 3) >> 2;
  const int64_t c = blockIdx.x / hg4;
  const int hv = static_cast<int>(blockIdx.x % hg4) * 4 + wid;
  if (c == p.NTmax) {
    // The one block past the chunks (N <= kWaveSeqs): the sequences by rank,
    // which the state kernel's blocks would otherwise each work out (a loop
    // over N in every wave), and the segment plan.
    if (wid > 0) return;
    const WaveSeqs w = wave_seqs(p);
    int rank = 0;
    for (int m = 0; m < static_cast<int>(p.N); ++m) {
      const int32_t cm = __builtin_amdgcn_readlane(w.cnt, m);
      rank += (cm > w.cnt) || (cm == w.cnt && m < lane);
    }
    if (lane < p.N)
      p.seqtab[rank] = make_int4(lane, w.incl - w.cnt, static_cast<int>(w.a), static_cast<int>(w.b));
    if (p.seg_max) {
      const int len = wave_seg_len(p);
      if (lane == 0) *p.seg_len = len;
    }
    return;
  }
  int64_t s;
  int L;
  if (p.N <= kWaveSeqs) {
    int64_t n;
    if (!wave_locate_chunk(p, c, n, s, L)) L = 0;
  } else {
    const int2 ce = p.ctab[c];  // (first token, length); length 0 past the last chunk
    s = ce.x;
    L = ce.y;
  }
  // Wave-uniform exit; the kernel has no block-level barriers.
  if (!(hv < p.HV && L > 0)) return;
  float (*X)[kLd] = lds[wid];
  float* gcv = vec[wid][0];
  float* btv = vec[wid][1];
  float* rkv = vec[wid][2];
  float* rqv = vec[wid][3];
  float* ckv = vec[wid][4];
  const int hq = hv / (p.HV / p.H);
  constexpr int KK = K / 32;
  const int64_t rs = p.sqk;

  // K rows of the chunk as MFMA operands (A and B^T read the same rows),
  // loaded quad-contiguously (q4_load; rows >= L repeat row L-1).  Every
  // product here pairs two such operands, so q4_to_a's key order needs no
  // change on the other side.
  static_assert(K == 128, "q4 operand loads are 16 x 128");
  const bf16* kbase = reinterpret_cast<const bf16*>(p.k) + static_cast<int64_t>(hq) * K;
  const bf16* qbase = reinterpret_cast<const bf16*>(p.q) + static_cast<int64_t>(hq) * K;
  bf8_t kop[4][KK];
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
    q4_load([&](int r) { return kbase + (s + min(mi * 16 + r, L - 1)) * rs; }, kop[mi]);
  // Per-token g (inclusive scan within the chunk) and beta; padded rows 0
  // (loads clamped to row L-1, then selected away).
  const int lt = min(lane, L - 1);
  const float graw = ldf<GT>(p.g, (s + lt) * p.HV + hv);
  const float braw = ldf<BT>(p.beta, (s + lt) * p.HV + hv);
  float gv = lane < L ? graw : 0.f;
  const float bv = lane < L ? braw : 0.f;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const float t = __shfl_up(gv, o, kWave);
    if (lane >= o) gv += t;
  }
  gcv[lane] = gv;
  btv[lane] = bv;
  // Row scales r = 1 / sqrt(sum x^2 + 1e-6) of the rows this lane holds
  // (row mi*16 + l15; the four lg lanes hold its four 32-wide pieces), or 1
  // without the in-op l2norm.
#pragma unroll
  for (int mi = 0; mi < 4; ++mi) q4_to_a(kop[mi]);
  row_scales<KK>(kop, rkv, p.l2norm);
  __builtin_amdgcn_wave_barrier();

  // The decay exp(gc_i - gc_j) of the tiles below the diagonal ones is a
  // product of factors of rows, columns and tiles, each <= 1 for decays <= 1
  // (an underflow of one underflows the product): with G_t = gc at the end
  // of 16-token block t - 1, row i of block mi and column j of block nj < mi,
  //   exp(gc_i - gc_j) = exp(gc_i - G_mi) exp(G_mi - G_{nj+1}) exp(G_{nj+1} - gc_j).
  // An element then takes two multiplies instead of an exponential and six
  // VALU instructions.  c_k = r_k exp(G_{nj+1} - gc) is formed once per token.
  // 24 of an M or Aq tile's 40 elements per lane; the kernel at 16,384 tokens
  // x 32 v-heads traced on one MI355X: 80.2 -> 78.2 us.
  ckv[lane] = rkv[lane] * __expf(gcv[lane | 15] - gv);
  float tile_decay[3];  // exp(G_mi - G_{nj+1}) of (2, 0), (3, 1), (3, 0)
  {
    const float g1 = readlane_f32(gv, 15), g2 = readlane_f32(gv, 31), g3 = readlane_f32(gv, 47);
    tile_decay[0] = __expf(g2 - g1);
    tile_decay[1] = __expf(g3 - g2);
    tile_decay[2] = __expf(g3 - g1);
  }
  auto tile_scale = [&](int mi, int nj) {
    return mi - nj == 1 ? 1.f : tile_decay[mi == 2 ? 0 : nj == 1 ? 1 : 2];
  };
  // exp(gc_i - G_mi) of the lane's row of block mi.
  auto row_decay = [&](int mi, float gr) { return mi ? __expf(gr - readlane_f32(gv, 16 * mi - 1)) : 1.f; };
  __builtin_amdgcn_wave_barrier();

  // M = strict_tril(b_i r_i r_j (k_i . k_j) exp(gc_i - gc_j)) into X (the
  // ten lower 16x16 tiles; the strictly upper ones are never read).  The
  // product K_nj K_mi^T is tile (mi, nj) transposed, so a lane holds row
  // mi*16 + l15, columns nj*16 + 4 lg .. + 3, written as one 16-byte vector.
#pragma unroll
  for (int mi = 0; mi < 4; ++mi) {
    const int row = mi * 16 + l15;
    const float fr = btv[row] * rkv[row], gr = gcv[row];
    const float fd = fr * row_decay(mi, gr);
#pragma unroll
    for (int nj = 0; nj <= mi; ++nj) {
      f4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) a = mfma16(kop[nj][kk], kop[mi][kk], a);
      f4_t m;
      if (nj < mi) {
        const f4_t ck = *reinterpret_cast<const f4_t*>(ckv + nj * 16 + 4 * lg);
        const float ft = fd * tile_scale(mi, nj);
#pragma unroll
        for (int i = 0; i < 4; ++i) m[i] = ft * ck[i] * a[i];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int col = nj * 16 + 4 * lg + i;
          m[i] = row > col ? fr * rkv[col] * a[i] * __expf(gr - gcv[col]) : 0.f;
        }
      }
      *reinterpret_cast<f4_t*>(&X[row][nj * 16 + 4 * lg]) = m;
    }
  }
  __builtin_amdgcn_wave_barrier();

  // Q rows, loaded before the inverse so that their latency hides behind
  // it (252 VGPRs with them live; the LDS footprint already limits the
  // kernel to two waves per SIMD, so the registers cost no occupancy).
  // Measured on MI355X at config 4: 87.6 -> 84.4 us.
  bf8_t qop[4][KK];
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
    q4_load([&](int r) { return qbase + (s + min(mi * 16 + r, L - 1)) * rs; }, qop[mi]);

  invert_unit_lower(X);  // X = (I + M)^-1, row-major

  char* rec = rec_at(p, c, hv);
  __bf16* aih = reinterpret_cast<__bf16*>(rec);
  __bf16* ail = reinterpret_cast<__bf16*>(rec + kMat);
  __bf16* aqp = reinterpret_cast<__bf16*>(rec + 2 * kMat);
  float* sc = reinterpret_cast<float*>(rec + 3 * kMat);
  // Ai as hi and lo bf16 operand images.  Store j writes image j, one
  // contiguous KB, so every store instruction writes whole cache lines;
  // image j = img_index(w, kk) for (w, kk) = (0,0) (1,0) (2,0) (2,1) (3,0)
  // (3,1).  Lane l reads X row 16 w + l % 16 from column 32 kk + 8 (l / 16):
  // 8 lanes of one b128 read cover all 32 banks (row stride 68 = 4 mod 32).
  auto tri_row = [&](int j) { return 16 * (j < 2 ? j : 2 + ((j - 2) >> 1)) + l15; };
  auto tri_col = [&](int j) { return 32 * (j < 2 ? 0 : (j - 2) & 1) + 8 * lg; };
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    bf8_t h, l;
    split8(&X[tri_row(j)][tri_col(j)], h, l);
    *reinterpret_cast<bf8_t*>(aih + 512 * j + 8 * lane) = h;
    *reinterpret_cast<bf8_t*>(ail + 512 * j + 8 * lane) = l;
  }
  __builtin_amdgcn_wave_barrier();

#pragma unroll
  for (int mi = 0; mi < 4; ++mi) q4_to_a(qop[mi]);
  row_scales<KK>(qop, rqv, p.l2norm);
  __builtin_amdgcn_wave_barrier();

  // Aq = scale * tril(r_q r_k (q k^T) exp(gc_i - gc_j)), rows < L, formed
  // transposed like M (K_nj Q_mi^T) for 16-byte row writes.
#pragma unroll
  for (int mi = 0; mi < 4; ++mi) {
    const int row = mi * 16 + l15;
    const float fr = row < L ? p.scale * rqv[row] : 0.f, gr = gcv[row];
    const float fd = fr * row_decay(mi, gr);
#pragma unroll
    for (int nj = 0; nj < 4; ++nj) {
      f4_t val = {0.f, 0.f, 0.f, 0.f};
      if (nj <= mi) {
        f4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) a = mfma16(kop[nj][kk], qop[mi][kk], a);
        if (nj < mi) {
          const f4_t ck = *reinterpret_cast<const f4_t*>(ckv + nj * 16 + 4 * lg);
          const float ft = fd * tile_scale(mi, nj);
#pragma unroll
          for (int i = 0; i < 4; ++i) val[i] = ft * ck[i] * a[i];
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int col = nj * 16 + 4 * lg + i;
            val[i] = row >= col ? fr * rkv[col] * a[i] * __expf(gr - gcv[col]) : 0.f;
          }
        }
      }
      *reinterpret_cast<f4_t*>(&X[row][nj * 16 + 4 * lg]) = val;
    }
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    bf8_t h;
#pragma unroll
    for (int e = 0; e < 8; ++e) h[e] = static_cast<__bf16>(X[tri_row(j)][tri_col(j) + e]);
    *reinterpret_cast<bf8_t*>(aqp + 512 * j + 8 * lane) = h;
  }

  // Per-token factors (lane = token); rows >= L are zero.
  const float gl = __shfl(gv, L - 1, kWave);
  const bool in = lane < L;
  const float eg = __expf(gv);
  sc[0 * kC + lane] = in ? p.scale * eg * rqv[lane] : 0.f;
  sc[1 * kC + lane] = in ? bv * eg * rkv[lane] : 0.f;
  sc[2 * kC + lane] = bv;
  sc[3 * kC + lane] = in ? rkv[lane] * __expf(gl - gv) : 0.f;
  sc[4 * kC + lane] = __expf(gl);
}

// ---------------------------------------------------------------------------
// P2: sequential chunk loop per (sequence, v-head, 32-column V tile), for V
// not a multiple of 64 (the 64-column kernel below covers the rest).
// ---------------------------------------------------------------------------
constexpr int kLt = kC + 8;  // bf16 LDS row stride (144 B: 16-byte aligned)

// The fp32 state tile itself lives in registers (each wave owns K/4 of its
// rows, in MFMA C layout); LDS holds its bf16 hi / lo copy, the B operand of
// K S, refreshed once per chunk.
template <int K, int BV>
struct __align__(16) P2Smem {
  __bf16 sb[2][BV][K + 8];    // state hi / lo, transposed: sb[h][v][k]
  __bf16 kr[2][kC * K];       // chunk key rows (kr_off layout), double-buffered
  __bf16 rt[2][BV][kLt];      // R transposed, hi / lo
  __bf16 vt[BV][kLt];         // Vn transposed (bf16, for the output)
  __bf16 dt[2][BV][kLt];      // (ed * Vn) transposed, hi / lo
};

// Operands one lane reads from global memory for one chunk, in three
// groups.  Those the chunk consumes first are double-buffered (loaded a whole
// chunk ahead).  The two later groups have one buffer each, refilled with
// the next chunk's operands right after their last use in the current chunk
// (so each load has most of a chunk to land) -- this keeps two waves per
// SIMD.
template <int KK, int NV32>
struct EarlyOps {
  bf8_t kA[KK];          // K rows wid*16.. as q4_load leaves them (stored as they are
                         // into the chunk's key tile, store_kr_q4)
  bf8_t vA[NV32];        // v row wid*16 + l15, tile columns 32j + 8*lg .. + 7
                         // (A layout; select_op turns it into C layout)
  f4_t ck, bt;           // factors of rows wid*16 + 4*lg + i
  float egl;             // exp(gc_last)
};
struct InvOps {          // consumed by Vn = Ai R and ed * Vn
  bf8_t aiH[2], aiL[2];  // Ai rows wid*16 + l15, hi / lo
  f4_t ed;
};
template <int KK>
struct OutOps {          // consumed by the output o = cq (Q S) + Aq Vn
  bf8_t qA[KK];          // Q rows wid*16.., as kA
  bf8_t aq[2];           // Aq rows wid*16 + l15
  float cq;              // factor of row wid*16 + l15
};

// Token row of q/k/v for C-layout row `r` (rows >= L read row L-1: finite,
// and zeroed by their factors).
template <int K, int BV>
__device__ __forceinline__ void load_early(const ChunkParams& p, EarlyOps<K / 32, BV / 32>& ops,
                                           int64_t s, int L, int64_t cidx, int hv, int hq,
                                           int vcol0) {
  const int lane = threadIdx.x & 63, wid = wave_index();
  const int l15 = lane & 15, lg = lane >> 4;
  const uint32_t rs = p.sqk;
  const WaveRows wr = wave_rows(s, L, wid);
  const char* kb = reinterpret_cast<const char*>(reinterpret_cast<const bf16*>(p.k) +
                                                 wr.row0 * rs + hq * K);
  q4_load_b(kb, 2 * rs, wr.lw, ops.kA);
  const char* vb = reinterpret_cast<const char*>(reinterpret_cast<const bf16*>(p.v) +
                                                 wr.row0 * p.sv + vcol0);
#pragma unroll
  for (int j = 0; j < BV / 32; ++j)
    ops.vA[j] = *reinterpret_cast<const bf8_t*>(vb + row_off(l15, wr.lw, 2 * p.sv, 32 * j + 8 * lg));
  const float* sc = reinterpret_cast<const float*>(rec_at(p, cidx, hv) + 3 * kMat);
  const int r4 = wid * 16 + 4 * lg;
  ops.ck = *reinterpret_cast<const f4_t*>(sc + 1 * kC + r4);
  ops.bt = *reinterpret_cast<const f4_t*>(sc + 2 * kC + r4);
  ops.egl = sc[4 * kC];
}

__device__ __forceinline__ void load_inv(const ChunkParams& p, InvOps& ops, int64_t cidx,
                                         int hv) {
  const int lane = threadIdx.x & 63, wid = wave_index();
  const int lg = lane >> 4;
  const char* rec = rec_at(p, cidx, hv);
  const float* sc = reinterpret_cast<const float*>(rec + 3 * kMat);
  // Rows 0..31 have no stored columns 32..63 (zero): their kk = 1 operand
  // re-reads the kk = 0 image, keeping every load unconditional, and is
  // never multiplied (the Vn product skips it).
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const char* img = rec + img_index(wid, kk) * 1024;
    ops.aiH[kk] = *reinterpret_cast<const bf8_t*>(img + 16 * lane);
    ops.aiL[kk] = *reinterpret_cast<const bf8_t*>(img + kMat + 16 * lane);
  }
  ops.ed = *reinterpret_cast<const f4_t*>(sc + 3 * kC + wid * 16 + 4 * lg);
}

template <int K>
__device__ __forceinline__ void load_out(const ChunkParams& p, OutOps<K / 32>& ops, int64_t s,
                                         int L, int64_t cidx, int hv, int hq) {
  const int lane = threadIdx.x & 63, wid = wave_index();
  const int l15 = lane & 15;
  const uint32_t rs = p.sqk;
  const WaveRows wr = wave_rows(s, L, wid);
  const char* qb = reinterpret_cast<const char*>(reinterpret_cast<const bf16*>(p.q) +
                                                 wr.row0 * rs + hq * K);
  q4_load_b(qb, 2 * rs, wr.lw, ops.qA);
  const char* rec = rec_at(p, cidx, hv);
  const float* sc = reinterpret_cast<const float*>(rec + 3 * kMat);
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)  // waves 0, 1: kk = 1 as for Ai
    ops.aq[kk] = *reinterpret_cast<const bf8_t*>(rec + 2 * kMat + img_index(wid, kk) * 1024 + 16 * lane);
  ops.cq = sc[0 * kC + wid * 16 + l15];
}

template <int K, typename T, int BV>
__global__ void __launch_bounds__(kTh) __attribute__((amdgpu_waves_per_eu(BV == 32 ? 2 : 1)))
gdn_chunk_state_kernel(ChunkParams p, int nvt) {
  static_assert(BV == 32 || BV == 64, "V tile of 32 or 64 columns");
  __shared__ P2Smem<K, BV> sm;
  constexpr int KK = K / 32;
  constexpr int NJ = BV / 16;  // 16-column tiles per block
  const int tid = threadIdx.x;
  const int wid = wave_index();
  const int lane = tid & 63;
  const int l15 = lane & 15, lg = lane >> 4;
  // XCD-aware mapping: the nvt V tiles of one (sequence, head) get block ids
  // that are equal modulo 8, i.e. run on the same XCD and share its L2.
  // Items are dispatched longest sequence first, so the longest chains start
  // in the first wave of resident blocks.
  const int64_t w = blockIdx.x;
  const int64_t xcd = w & 7, r = w >> 3;
  const int vt = static_cast<int>(r % nvt);
  const int64_t item = (r / nvt) * 8 + xcd;  // (sequence rank, head) index
  if (item >= p.N * p.HV) return;            // whole block
  const SeqEntry se = ranked_seq(p, item / p.HV);
  const int64_t n = se.n, cidx0 = se.c0, bos = se.bos, eos = se.eos;
  const int hv = state_head(static_cast<int>(item % p.HV), p.HV, p.H);
  const int hq = hv / (p.HV / p.H);
  const int V = nvt * BV;
  const int v0 = vt * BV;
  // Chunks of this sequence; the NTmax bound keeps a malformed cu_seqlens
  // (never a well-formed one) from reading past the workspace.
  const int64_t nch = max<int64_t>(0, min<int64_t>((eos - bos + kC - 1) / kC, p.NTmax - cidx0));

  // State rows (k) wid*(K/4) + m2*16 + 4*lg + i, columns nj*16 + l15.
  constexpr int M2 = K / 64;
  f4_t sreg[M2][NJ];
#pragma unroll
  for (int m2 = 0; m2 < M2; ++m2)
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int kr = wid * (K / 4) + m2 * 16 + 4 * lg + i;
        sreg[m2][nj][i] = p.h0 ? p.h0[((n * p.HV + hv) * K + kr) * V + v0 + nj * 16 + l15] : 0.f;
      }
  // bf16 hi / lo copy of the state for the K S operand.
  auto publish_state = [&]() {
#pragma unroll
    for (int m2 = 0; m2 < M2; ++m2)
#pragma unroll
      for (int nj = 0; nj < NJ; ++nj) {
        Vec<__bf16, 4> h, l;
        split4(sreg[m2][nj], h, l);
        const int k0 = wid * (K / 4) + m2 * 16 + 4 * lg;
        *reinterpret_cast<Vec<__bf16, 4>*>(&sm.sb[0][nj * 16 + l15][k0]) = h;
        *reinterpret_cast<Vec<__bf16, 4>*>(&sm.sb[1][nj * 16 + l15][k0]) = l;
      }
  };
  publish_state();
  const uint32_t vrow = static_cast<uint32_t>(p.HV) * V;  // o token stride
  const int vcol0 = hv * V + v0;
  const bf8_t sel[2] = {select_op(0), select_op(1)};
  EarlyOps<KK, BV / 32> opsA, opsB;
  InvOps inv;
  OutOps<KK> outo;
  if (nch > 0) {
    const int L0 = static_cast<int>(min<int64_t>(kC, eos - bos));
    load_early<K, BV>(p, opsA, bos, L0, cidx0, hv, hq, vcol0);
    // Keep the early group ahead of the others, in loop order: the loop's
    // wait counts are fixed by the shortest distance (in memory operations)
    // between a load and its first use over every path, this one included,
    // and an early load scheduled last here would make every chunk wait for
    // the previous chunk's most recent loads.
    __builtin_amdgcn_sched_barrier(0);
    load_inv(p, inv, cidx0, hv);
    __builtin_amdgcn_sched_barrier(0);
    load_out<K>(p, outo, bos, L0, cidx0, hv, hq);
    store_kr_q4(sm.kr[0], opsA.kA, wid);
  }
  __syncthreads();

  // One chunk: `cur` holds its early operands, `nxt` receives the next
  // chunk's; `inv` and `outo` are refilled with the next chunk's operands
  // right after their last use here.  The last chunk "prefetches" itself
  // again (unused), so that every memory operation of the loop is
  // unconditional.
  auto step = [&](const EarlyOps<KK, BV / 32>& cur, EarlyOps<KK, BV / 32>& nxt, int64_t ci) {
    const int64_t s = bos + ci * kC;
    const int L = static_cast<int>(min<int64_t>(kC, eos - s));
    const int64_t cn = min(ci + 1, nch - 1);
    const int64_t sn = bos + cn * kC;
    const int Ln = static_cast<int>(min<int64_t>(kC, eos - sn));
    load_early<K, BV>(p, nxt, sn, Ln, cidx0 + cn, hv, hq, vcol0);

    // KS = K S (hi/lo S): rows wid*16.., columns nj*16..; K's rows come
    // from the chunk's key tile.
    const __bf16* kr = sm.kr[ci & 1];
    f4_t ks[NJ];
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj) ks[nj] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const bf8_t ka = kr_a(kr, wid, kk);
#pragma unroll
      for (int nj = 0; nj < NJ; ++nj) {
        const bf8_t sh = *reinterpret_cast<const bf8_t*>(&sm.sb[0][nj * 16 + l15][kk * 32 + 8 * lg]);
        const bf8_t sl = *reinterpret_cast<const bf8_t*>(&sm.sb[1][nj * 16 + l15][kk * 32 + 8 * lg]);
        ks[nj] = mfma16(ka, sh, ks[nj]);
        ks[nj] = mfma16(ka, sl, ks[nj]);
      }
    }
    // R = b v - ck KS  ->  rt (transposed, hi / lo); padded rows are 0.
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj) {
      Vec<__bf16, 4> h, l;
      const f4_t vc = mfma16(cur.vA[nj >> 1], sel[nj & 1], f4_t{0.f, 0.f, 0.f, 0.f});
      f4_t rv;
#pragma unroll
      for (int i = 0; i < 4; ++i) rv[i] = cur.bt[i] * vc[i] - cur.ck[i] * ks[nj][i];
      split4(rv, h, l);
      *reinterpret_cast<Vec<__bf16, 4>*>(&sm.rt[0][nj * 16 + l15][wid * 16 + 4 * lg]) = h;
      *reinterpret_cast<Vec<__bf16, 4>*>(&sm.rt[1][nj * 16 + l15][wid * 16 + 4 * lg]) = l;
    }
    __syncthreads();  // (1) rt complete

    // Vn = Ai R.
    f4_t vn[NJ];
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj) {
      vn[nj] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        if (kk * 32 > wid * 16 + 15) continue;  // zero block of Ai (not stored)
        const bf8_t rh = *reinterpret_cast<const bf8_t*>(&sm.rt[0][nj * 16 + l15][kk * 32 + 8 * lg]);
        const bf8_t rl = *reinterpret_cast<const bf8_t*>(&sm.rt[1][nj * 16 + l15][kk * 32 + 8 * lg]);
        vn[nj] = mfma_split3(inv.aiH[kk], inv.aiL[kk], rh, rl, vn[nj]);
      }
    }
    // Vn -> vt (bf16), ed * Vn -> dt (hi / lo).
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj) {
      Vec<__bf16, 4> b, h, l;
      f4_t d;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        b.v[i] = static_cast<__bf16>(vn[nj][i]);
        d[i] = inv.ed[i] * vn[nj][i];
      }
      split4(d, h, l);
      *reinterpret_cast<Vec<__bf16, 4>*>(&sm.vt[nj * 16 + l15][wid * 16 + 4 * lg]) = b;
      *reinterpret_cast<Vec<__bf16, 4>*>(&sm.dt[0][nj * 16 + l15][wid * 16 + 4 * lg]) = h;
      *reinterpret_cast<Vec<__bf16, 4>*>(&sm.dt[1][nj * 16 + l15][wid * 16 + 4 * lg]) = l;
    }
    load_inv(p, inv, cidx0 + cn, hv);  // this chunk is done with `inv`
    // (Q S)^T = S^T Q^T with the hi part of S: the output is produced
    // transposed (lane: token wid*16 + l15, columns 4*lg .. 4*lg + 3), so
    // each lane stores one 8-byte vector per column tile.  The S^T A operand
    // is the same sb read as S's B operand, and Q^T's B operand is Q's A
    // operand.  It must read sb before barrier 2: after it, a wave that is
    // ahead may already publish the next state into sb.
    q4_to_a(outo.qA);
    f4_t qs[NJ];
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj) {
      qs[nj] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        const bf8_t sh = *reinterpret_cast<const bf8_t*>(&sm.sb[0][nj * 16 + l15][q4_key(kk, lg)]);
        qs[nj] = mfma16(sh, outo.qA[kk], qs[nj]);
      }
    }
    __syncthreads();  // (2) vt, dt complete; rt and sb reads done

    // o^T = cq (Q S)^T + Vn^T Aq^T (Vn^T's A operand is the vt read that
    // was Vn's B operand; Aq^T's B operand is Aq's A operand).
    // The MFMA leaves lane (g = lane / 16, t = lane % 16) with row t,
    // columns nj*16 + 4 g ..; before the store, lane (r = lane / 16, a =
    // lane / 4 % 4, b = lane % 4) pulls (ds_bpermute) the values of row
    // 4 a + r, column group b from lane 16 b + 4 a + r.  Each quad then
    // writes 32 contiguous bytes of one row, where the MFMA layout had the 4
    // lanes of a quad write 4 different rows (7 us of the state kernel at
    // config 4 on MI355X).
    static_assert(sizeof(T) == 2, "two dwords per 4-column group");
    {
      const int row = wid * 16 + quad_row(), qb = quad_col();
      T* orow = row < L ? reinterpret_cast<T*>(p.o) + static_cast<uint64_t>(s + row) * vrow + vcol0
                        : reinterpret_cast<T*>(p.dump) + row * BV;
#pragma unroll
      for (int nj = 0; nj < NJ; ++nj) {
        f4_t acc;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = outo.cq * qs[nj][i];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          if (kk * 32 > wid * 16 + 15) continue;  // Aq columns beyond the diagonal
          const bf8_t vb = *reinterpret_cast<const bf8_t*>(&sm.vt[nj * 16 + l15][kk * 32 + 8 * lg]);
          acc = mfma16(vb, outo.aq[kk], acc);
        }
        Vec<T, 4> ov;
#pragma unroll
        for (int i = 0; i < 4; ++i) ov.v[i] = from_f32<T>(acc[i]);
        *reinterpret_cast<u32x2*>(orow + nj * 16 + 4 * qb) = quad_rows(__builtin_bit_cast(u32x2, ov));
      }
    }
    load_out<K>(p, outo, sn, Ln, cidx0 + cn, hv, hq);  // this chunk is done with `outo`

    // S <- exp(gc_last) S + K^T (ed Vn) on the wave's register rows, then
    // its bf16 copy (every wave finished reading sb before barrier 2).
#pragma unroll
    for (int m2 = 0; m2 < M2; ++m2) {
      const int mi = wid * M2 + m2;
      bf8_t ka[2];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) ka[kk] = kr_at(kr, mi, kk);
#pragma unroll
      for (int nj = 0; nj < NJ; ++nj) {
        f4_t acc = sreg[m2][nj];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] *= cur.egl;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          const bf8_t dh = *reinterpret_cast<const bf8_t*>(&sm.dt[0][nj * 16 + l15][kk * 32 + 8 * lg]);
          const bf8_t dl = *reinterpret_cast<const bf8_t*>(&sm.dt[1][nj * 16 + l15][kk * 32 + 8 * lg]);
          acc = mfma16(ka[kk], dh, acc);
          acc = mfma16(ka[kk], dl, acc);
        }
        sreg[m2][nj] = acc;
      }
    }
    publish_state();
    store_kr_q4(sm.kr[(ci + 1) & 1], nxt.kA, wid);
    __syncthreads();  // (3) state copy, next keys complete; vt / dt / key reads done
  };
  // Unrolled by two so the operand buffers swap roles without copies.
  for (int64_t ci = 0; ci < nch; ci += 2) {
    step(opsA, opsB, ci);
    if (ci + 1 < nch) step(opsB, opsA, ci + 1);
  }
  if (p.ht) {
#pragma unroll
    for (int m2 = 0; m2 < M2; ++m2)
#pragma unroll
      for (int nj = 0; nj < NJ; ++nj)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int kr = wid * (K / 4) + m2 * 16 + 4 * lg + i;
          p.ht[((n * p.HV + hv) * K + kr) * V + v0 + nj * 16 + l15] = sreg[m2][nj][i];
        }
  }
}

// ---------------------------------------------------------------------------
// P2 with one 512-lane block per (sequence, v-head, 64-column V tile): eight
// waves, wave (wr = wid % 4, cg = wid / 4) owning token rows 16 wr .., state
// key rows 32 wr .. and columns 32 cg .. of the tile, exactly the share of a
// wave of gdn_chunk_state_kernel.  The two column groups share the chunk's
// key and query rows: each wave loads 8 of the 64 rows of each as whole
// rows, into a key tile (read as rows for K S and transposed for the state
// update) and a query tile (read as rows for Q S, so Q needs no register
// transpose).  One block per CU (132 KB of LDS), two waves per SIMD as with
// two 256-lane blocks; the loop issues 31% fewer VALU instructions than the
// 256-lane kernel's.  Measured on MI355X at config 4: 226.8 -> 221.6 us.
// The per-token factors (cq, ck, beta, ed) reach the waves through a 1 KB
// LDS tile that every wave fills with one load of the record's factor
// block, instead of four loads of its own rows of them; e^{g_last} is a
// scalar load.  That is 4 fewer vector-memory instructions per wave and
// step and 24 fewer VGPRs (222 -> 198): 223.9 -> 221.5 us.
// ---------------------------------------------------------------------------
constexpr int kTh8 = 512;

// Modes of the 64-column state kernel: whole sequences, or (segments of a
// sequence in parallel) end states and transitions only, then outputs.
enum { kSegNone = 0, kSegSum = 1, kSegOut = 2 };

// The transposed tiles below (sb8_off, t8_off) are unpadded and swizzled.

template <int K>
struct __align__(16) P2Smem8 {
  __bf16 sb[2][64 * K];     // state hi / lo, transposed: [v][k] (sb8_off)
  __bf16 kr[2][kC * K];     // chunk key rows (kr_off layout), double-buffered
  __bf16 qr[kC * K];        // chunk query rows (kr_off layout)
  __bf16 rt[2][64 * kC];    // R transposed, hi / lo (t8_off)
  __bf16 vt[64 * kC];       // Vn transposed (bf16, for the output)
  __bf16 dt[2][64 * kC];    // (ed * Vn) transposed, hi / lo
  float fac[2][4 * kC];     // per-token factors cq, ck, beta, ed of the chunk, double-buffered
};

struct EarlyOps8 {
  bf8_t kraw[2], qraw[2];  // key / query rows 16 wr + 8 cg + 4 j + lane / 16, chunk lane % 16
  bf8_t vA;                // v row 16 wr + l15, columns 32 cg + 8 lg .. + 7 (A layout)
  f4_t fac;                // factor floats 4 lane .. 4 lane + 3 of the record
  float egl;
};
struct InvOps8 {
  bf8_t aiH[2], aiL[2];
};
struct OutOps8 {
  bf8_t aq[2];
};
typedef __attribute__((address_space(4))) const float cfloat_t;

template <int K, int MODE>
__global__ void __launch_bounds__(kTh8) __attribute__((amdgpu_waves_per_eu(2)))
gdn_chunk_state8_kernel(ChunkParams p, int nvt) {
  constexpr int BV = 64;
  static_assert(K == 128, "key rows of 128");
  __shared__ P2Smem8<K> sm;
  constexpr int KK = K / 32;
  constexpr int NJ = 2;  // 16-column tiles per wave
  constexpr bool kOut = MODE != kSegSum;
  const int tid = threadIdx.x;
  const int wid = wave_index();
  // Waves w and w + 4 share a SIMD; they take token rows wr and 3 - wr, so
  // that every SIMD gets the same share of the triangular products (Ai and
  // Aq hold 1, 1, 2, 2 nonzero 32-wide pieces for rows 0..3).  Measured on
  // MI355X at config 4: 283.0 -> 280.1 us per call.
  const int cg = wid >> 2, wr = cg ? 3 - (wid & 3) : (wid & 3), cb = 32 * cg;
  const int lane = tid & 63;
  const int l15 = lane & 15, lg = lane >> 4;
  const int rl = lane >> 4, ch = lane & 15;  // whole-row loads: row in a load, 16-byte chunk
  const int64_t w = blockIdx.x;
  const int64_t xcd = w & 7, r = w >> 3;
  const int ntile = MODE == kSegSum ? nvt + K / 64 : nvt;
  const int vt = static_cast<int>(r % ntile);
  const int64_t item = (r / ntile) * 8 + xcd;
  const int hv = state_head(static_cast<int>(item % p.HV), p.HV, p.H);
  const int hq = hv / (p.HV / p.H);
  const int V = nvt * BV;
  const bool is_m = MODE == kSegSum && vt >= nvt;  // block of the transition's columns
  const int v0 = is_m ? 0 : vt * BV;
  int64_t n, cidx0, bos, eos, nch;
  // Where the state comes from (NULL: zero) and goes to (NULL: nowhere).
  const float* s_in;
  float* s_out;
  int64_t sh = 0;  // (segment, head)
  int before = 0;  // segments of the sequence before this one
  if constexpr (MODE == kSegNone) {
    if (item >= p.N * p.HV) return;
    const SeqEntry se = ranked_seq(p, item / p.HV);
    n = se.n;
    cidx0 = se.c0;
    bos = se.bos;
    eos = se.eos;
    nch = (eos - bos + kC - 1) / kC;
    const int64_t at = (n * p.HV + hv) * K * V;
    s_in = p.h0 ? p.h0 + at : nullptr;
    s_out = p.ht ? p.ht + at : nullptr;
  } else {
    if (MODE == kSegSum && !*p.seg_len) return;  // (with 1 block a CU, idle ones should be short)
    const WaveSegs ws = wave_segs(p);
    // kSegSum blocks skip the last segment of every sequence: its end state
    // is not needed.
    const int skip = MODE == kSegSum ? (lane < p.N ? lane + 1 : static_cast<int>(p.N)) : 0;
    const int64_t at_seg = item / p.HV;
    if (at_seg >= __builtin_amdgcn_readlane(ws.incl - skip, kWave - 1)) return;
    const int nn = __popcll(__ballot(ws.incl - skip <= at_seg));
    n = nn;
    const int cnt = __builtin_amdgcn_readlane(ws.cnt, nn);
    const int64_t seg = at_seg + (MODE == kSegSum ? nn : 0);
    if (seg >= p.seg_max) return;
    before = static_cast<int>(seg) - (__builtin_amdgcn_readlane(ws.incl, nn) - cnt);
    const int first = before * ws.len;  // chunk of the sequence
    sh = seg * p.HV + hv;
    cidx0 = __builtin_amdgcn_readlane(ws.s.incl - ws.s.cnt, nn) + first;
    bos = readlane64(ws.s.a, nn) + static_cast<int64_t>(first) * kC;
    eos = readlane64(ws.s.b, nn);
    nch = __builtin_amdgcn_readlane(ws.s.cnt, nn) - first;
    if (ws.len) nch = min(nch, ws.len);
    const int64_t at = (n * p.HV + hv) * K * V;
    s_in = p.h0 ? p.h0 + at : nullptr;
    if constexpr (MODE == kSegSum) {
      if (is_m && before == 0) return;  // the first segment's transition is not needed
      if (before > 0) s_in = nullptr;
      s_out = is_m ? nullptr : p.seg_b + sh * K * V;
    } else {
      const bool in_order = cnt > 1 && p.seg_bad[n * p.HV + hv] != 0;
      if (in_order) {
        if (before > 0) return;
        nch = __builtin_amdgcn_readlane(ws.s.cnt, nn);
      }
      if (before > 0) s_in = p.seg_b + (sh - p.HV) * K * V;
      s_out = p.ht && (in_order || before == cnt - 1) ? p.ht + at : nullptr;
    }
  }
  // The NTmax bound keeps a malformed cu_seqlens (never a well-formed one)
  // from reading past the workspace.
  nch = max<int64_t>(0, min<int64_t>(nch, p.NTmax - cidx0));
  const int scol = is_m ? (vt - nvt) * BV : vt * BV;  // first column of the state block

  constexpr int M2 = K / 64;
  const uint32_t vrow = static_cast<uint32_t>(p.HV) * V;
  const int vcol0 = hv * V + v0 + cb;
  const uint32_t rb = p.sqk * 2;  // q / k row pitch in bytes
  const bf8_t sel[2] = {select_op(0), select_op(1)};

  auto load_early8 = [&](EarlyOps8& o, int64_t s, int L, int64_t cidx) {
    const char* kb = reinterpret_cast<const char*>(reinterpret_cast<const bf16*>(p.k) + s * p.sqk + hq * K);
    const char* qb = reinterpret_cast<const char*>(reinterpret_cast<const bf16*>(p.q) + s * p.sqk + hq * K);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint32_t off = static_cast<uint32_t>(min(wr * 16 + cg * 8 + 4 * j + rl, L - 1)) * rb + 16u * ch;
      o.kraw[j] = *reinterpret_cast<const bf8_t*>(kb + off);
      if constexpr (kOut) o.qraw[j] = *reinterpret_cast<const bf8_t*>(qb + off);
    }
    const WaveRows wrs = wave_rows(s, L, wr);
    const char* vb = reinterpret_cast<const char*>(reinterpret_cast<const bf16*>(p.v) +
                                                   wrs.row0 * p.sv + vcol0);
    o.vA = *reinterpret_cast<const bf8_t*>(vb + row_off(l15, wrs.lw, 2 * p.sv, 8 * lg));
    if (is_m) o.vA = bf8_t{};  // a transition has no values (and takes no NaN from them)
    // The factor block (cq, ck, beta, ed: 1 KB) in one load per wave; the
    // wave-uniform e^{g_last} through the scalar cache.
    const char* sc = rec_at(p, cidx, hv) + 3 * kMat;
    o.fac = *reinterpret_cast<const f4_t*>(sc + 16 * lane);
    o.egl = *(cfloat_t*)(sc + 16 * kC);
  };
  auto load_inv8 = [&](InvOps8& o, int64_t cidx) {
    const char* rec = rec_at(p, cidx, hv);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const char* img = rec + img_index(wr, kk) * 1024;
      o.aiH[kk] = *reinterpret_cast<const bf8_t*>(img + 16 * lane);
      o.aiL[kk] = *reinterpret_cast<const bf8_t*>(img + kMat + 16 * lane);
    }
  };
  auto load_out8 = [&](OutOps8& o, int64_t cidx) {
    const char* rec = rec_at(p, cidx, hv);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
      o.aq[kk] = *reinterpret_cast<const bf8_t*>(rec + 2 * kMat + img_index(wr, kk) * 1024 + 16 * lane);
  };
  // Every wave writes the same factor bytes (one 16-byte store per lane).
  auto store_fac = [&](float* f, const f4_t& v) { *reinterpret_cast<f4_t*>(f + 4 * lane) = v; };
  auto store_rows = [&](__bf16* tile, const bf8_t (&raw)[2]) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
      *reinterpret_cast<bf8_t*>(tile + kr_off(wr * 16 + cg * 8 + 4 * j + rl, ch)) = raw[j];
  };

  EarlyOps8 opsA, opsB;
  InvOps8 inv;
  OutOps8 outo;
  // The first chunk's operands are requested before the initial state, so
  // that a block of a few chunks waits once.
  if (nch > 0) {
    const int L0 = static_cast<int>(min<int64_t>(kC, eos - bos));
    load_early8(opsA, bos, L0, cidx0);
    __builtin_amdgcn_sched_barrier(0);
    load_inv8(inv, cidx0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kOut) load_out8(outo, cidx0);
    __builtin_amdgcn_sched_barrier(0);
  }
  f4_t sreg[M2][NJ];
#pragma unroll
  for (int m2 = 0; m2 < M2; ++m2)
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int kr = wr * (K / 4) + m2 * 16 + 4 * lg + i;
        const int col = scol + cb + nj * 16 + l15;
        if (is_m) sreg[m2][nj][i] = kr == col ? 1.f : 0.f;
        else sreg[m2][nj][i] = s_in ? s_in[static_cast<int64_t>(kr) * V + col] : 0.f;
      }
  auto publish_state = [&]() {
#pragma unroll
    for (int m2 = 0; m2 < M2; ++m2)
#pragma unroll
      for (int nj = 0; nj < NJ; ++nj) {
        Vec<__bf16, 4> h, l;
        split4(sreg[m2][nj], h, l);
        const int k0 = wr * (K / 4) + m2 * 16 + 4 * lg;
        *reinterpret_cast<Vec<__bf16, 4>*>(&sm.sb[0][sb8_off(cb + nj * 16 + l15, k0)]) = h;
        *reinterpret_cast<Vec<__bf16, 4>*>(&sm.sb[1][sb8_off(cb + nj * 16 + l15, k0)]) = l;
      }
  };
  publish_state();
  if (nch > 0) {
    store_rows(sm.kr[0], opsA.kraw);
    if constexpr (kOut) store_rows(sm.qr, opsA.qraw);
    store_fac(sm.fac[0], opsA.fac);
  }
  __syncthreads();
  float decay = 1.f;  // kSegSum: product of the chunks' e^{g_last}, rounded as the state's is

  auto step = [&](const EarlyOps8& cur, EarlyOps8& nxt, int64_t ci) {
    const int64_t s = bos + ci * kC;
    const int L = static_cast<int>(min<int64_t>(kC, eos - s));
    const int64_t cn = min(ci + 1, nch - 1);
    const int64_t sn = bos + cn * kC;
    const int Ln = static_cast<int>(min<int64_t>(kC, eos - sn));
    load_early8(nxt, sn, Ln, cidx0 + cn);

    const __bf16* kr = sm.kr[ci & 1];
    const float* fc = sm.fac[ci & 1];
    const f4_t ck = *reinterpret_cast<const f4_t*>(fc + 1 * kC + wr * 16 + 4 * lg);
    const f4_t bt = *reinterpret_cast<const f4_t*>(fc + 2 * kC + wr * 16 + 4 * lg);
    f4_t ks[NJ];
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj) ks[nj] = f4_t{0.f, 0.f, 0.f, 0.f};
    // The scheduler's small-GEMM interleaving of LDS reads and MFMAs for the
    // K S and state-update products: 221.6 -> 216.6 us at config 4 on MI355X
    // (the variant for wider tiles, iglp_opt(1), took 237 us).
    __builtin_amdgcn_iglp_opt(0);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const bf8_t ka = kr_a(kr, wr, kk);
#pragma unroll
      for (int nj = 0; nj < NJ; ++nj) {
        const bf8_t sh = *reinterpret_cast<const bf8_t*>(&sm.sb[0][sb8_off(cb + nj * 16 + l15, kk * 32 + 8 * lg)]);
        const bf8_t sl = *reinterpret_cast<const bf8_t*>(&sm.sb[1][sb8_off(cb + nj * 16 + l15, kk * 32 + 8 * lg)]);
        ks[nj] = mfma16(ka, sh, ks[nj]);
        ks[nj] = mfma16(ka, sl, ks[nj]);
      }
    }
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj) {
      Vec<__bf16, 4> h, l;
      const f4_t vc = mfma16(cur.vA, sel[nj], f4_t{0.f, 0.f, 0.f, 0.f});
      f4_t rv;
#pragma unroll
      for (int i = 0; i < 4; ++i) rv[i] = bt[i] * vc[i] - ck[i] * ks[nj][i];
      split4(rv, h, l);
      *reinterpret_cast<Vec<__bf16, 4>*>(&sm.rt[0][t8_off(cb + nj * 16 + l15, wr * 16 + 4 * lg)]) = h;
      *reinterpret_cast<Vec<__bf16, 4>*>(&sm.rt[1][t8_off(cb + nj * 16 + l15, wr * 16 + 4 * lg)]) = l;
    }
    __syncthreads();  // (1)

    const f4_t ed = *reinterpret_cast<const f4_t*>(fc + 3 * kC + wr * 16 + 4 * lg);
    f4_t vn[NJ];
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj) {
      vn[nj] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        if (kk * 32 > wr * 16 + 15) continue;
        const bf8_t rh = *reinterpret_cast<const bf8_t*>(&sm.rt[0][t8_off(cb + nj * 16 + l15, kk * 32 + 8 * lg)]);
        const bf8_t rl2 = *reinterpret_cast<const bf8_t*>(&sm.rt[1][t8_off(cb + nj * 16 + l15, kk * 32 + 8 * lg)]);
        vn[nj] = mfma_split3(inv.aiH[kk], inv.aiL[kk], rh, rl2, vn[nj]);
      }
    }
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj) {
      Vec<__bf16, 4> b, h, l;
      f4_t d;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        b.v[i] = static_cast<__bf16>(vn[nj][i]);
        d[i] = ed[i] * vn[nj][i];
      }
      split4(d, h, l);
      if constexpr (kOut)
        *reinterpret_cast<Vec<__bf16, 4>*>(&sm.vt[t8_off(cb + nj * 16 + l15, wr * 16 + 4 * lg)]) = b;
      *reinterpret_cast<Vec<__bf16, 4>*>(&sm.dt[0][t8_off(cb + nj * 16 + l15, wr * 16 + 4 * lg)]) = h;
      *reinterpret_cast<Vec<__bf16, 4>*>(&sm.dt[1][t8_off(cb + nj * 16 + l15, wr * 16 + 4 * lg)]) = l;
    }
    load_inv8(inv, cidx0 + cn);
    // (Q S)^T = S^T Q^T: Q's rows from the query tile, keys in natural order.
    f4_t qs[NJ];
    if constexpr (kOut) {
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj) qs[nj] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const bf8_t qa = kr_a(sm.qr, wr, kk);
#pragma unroll
      for (int nj = 0; nj < NJ; ++nj) {
        const bf8_t sh = *reinterpret_cast<const bf8_t*>(&sm.sb[0][sb8_off(cb + nj * 16 + l15, kk * 32 + 8 * lg)]);
        qs[nj] = mfma16(sh, qa, qs[nj]);
      }
    }
    }
    __syncthreads();  // (2) vt, dt complete; rt, sb and query reads done

    if constexpr (kOut) {
      const int row = wr * 16 + quad_row(), qb = quad_col();
      const float cq = fc[0 * kC + wr * 16 + l15];
      bf16* orow = row < L ? reinterpret_cast<bf16*>(p.o) + static_cast<uint64_t>(s + row) * vrow + vcol0
                           : reinterpret_cast<bf16*>(p.dump) + row * BV + cb;
#pragma unroll
      for (int nj = 0; nj < NJ; ++nj) {
        f4_t acc;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = cq * qs[nj][i];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          if (kk * 32 > wr * 16 + 15) continue;
          const bf8_t vb = *reinterpret_cast<const bf8_t*>(&sm.vt[t8_off(cb + nj * 16 + l15, kk * 32 + 8 * lg)]);
          acc = mfma16(vb, outo.aq[kk], acc);
        }
        Vec<bf16, 4> ov;
#pragma unroll
        for (int i = 0; i < 4; ++i) ov.v[i] = from_f32<bf16>(acc[i]);
        *reinterpret_cast<u32x2*>(orow + nj * 16 + 4 * qb) = quad_rows(__builtin_bit_cast(u32x2, ov));
      }
    }
    if constexpr (kOut) load_out8(outo, cidx0 + cn);
    if constexpr (!kOut) decay *= cur.egl;

    __builtin_amdgcn_iglp_opt(0);
#pragma unroll
    for (int m2 = 0; m2 < M2; ++m2) {
      const int mi = wr * M2 + m2;
      bf8_t ka[2];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) ka[kk] = kr_at(kr, mi, kk);
#pragma unroll
      for (int nj = 0; nj < NJ; ++nj) {
        f4_t acc = sreg[m2][nj];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] *= cur.egl;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          const bf8_t dh = *reinterpret_cast<const bf8_t*>(&sm.dt[0][t8_off(cb + nj * 16 + l15, kk * 32 + 8 * lg)]);
          const bf8_t dl = *reinterpret_cast<const bf8_t*>(&sm.dt[1][t8_off(cb + nj * 16 + l15, kk * 32 + 8 * lg)]);
          acc = mfma16(ka[kk], dh, acc);
          acc = mfma16(ka[kk], dl, acc);
        }
        sreg[m2][nj] = acc;
      }
    }
    publish_state();
    store_rows(sm.kr[(ci + 1) & 1], nxt.kraw);
    if constexpr (kOut) store_rows(sm.qr, nxt.qraw);
    store_fac(sm.fac[(ci + 1) & 1], nxt.fac);
    __syncthreads();  // (3)
  };
  for (int64_t ci = 0; ci < nch; ci += 2) {
    step(opsA, opsB, ci);
    if (ci + 1 < nch) step(opsB, opsA, ci + 1);
  }
  if (is_m) {
    // M - c I, columns scol .. + 63, as A operands of the combine kernel, each
    // value in three bf16 parts: image (w, q, part) holds rows 16 w + l % 16
    // and, in the 16 bytes of lane l, columns 32 q + 4 (l / 16) + {0 .. 3, 16
    // .. 19}.  Quads transpose their 4 x 4 blocks of the MFMA layout for it.
    bool over = !(fabsf(decay) <= kSegLimit);
#pragma unroll
    for (int m2 = 0; m2 < M2; ++m2) {
      bf8_t part[3];
#pragma unroll
      for (int nj = 0; nj < NJ; ++nj) {
        f4_t x = sreg[m2][nj];
        const int kr = wr * (K / 4) + m2 * 16 + 4 * lg, col = scol + cb + nj * 16 + l15;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (kr + i == col) x[i] -= decay;
          over |= !(fabsf(x[i]) <= kSegLimit);
        }
        Vec<__bf16, 4> t[3];
        split4x3(quad_transpose(x), t);
#pragma unroll
        for (int u = 0; u < 3; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) part[u][4 * nj + i] = t[u].v[i];
      }
      char* img = p.seg_m + sh * kSegImg + ((wr * M2 + m2) * KK + (scol + cb) / 32) * 3072 +
                  16 * (16 * (l15 >> 2) + 4 * lg + (lane & 3));
#pragma unroll
      for (int u = 0; u < 3; ++u) *reinterpret_cast<bf8_t*>(img + 1024 * u) = part[u];
    }
    const int any = __syncthreads_or(over);
    if (tid == 0) {
      p.seg_over[2 * sh + (vt - nvt)] = any;
      if (vt == nvt) p.seg_c[sh] = decay;
    }
  } else if (s_out) {
#pragma unroll
    for (int m2 = 0; m2 < M2; ++m2)
#pragma unroll
      for (int nj = 0; nj < NJ; ++nj)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int kr = wr * (K / 4) + m2 * 16 + 4 * lg + i;
          s_out[static_cast<int64_t>(kr) * V + scol + cb + nj * 16 + l15] = sreg[m2][nj][i];
        }
  }
}


// ---------------------------------------------------------------------------
// States at the segment boundaries of one (sequence, v-head, 16 V columns):
// S_1 = the state after segment 0, S_{i+1} = c_i S_i + (M_i - c_i I) S_i +
// B_i; S_{i+1} replaces B_i.  A block of eight waves; wave w owns state rows
// 16 w .. + 15.  Both factors of the product enter in three bf16 parts, so it
// is good to 2^-24 (see "Segments").  A step waits for its 96 KB of operand
// images, read 2 to 3 us ahead into registers: 1.4 us (two parts: 64 KB and
// 1.0 us, but 2^-17; fp32 images and MFMA: 64 KB, 2.0 us of matrix time).
// Two steps in flight instead of three take 1.7 us a step.
// ---------------------------------------------------------------------------
template <int K>
__global__ void __launch_bounds__(kTh8) gdn_chunk_combine_kernel(ChunkParams p, int V) {
  static_assert(K == 128, "eight waves of 16 rows");
  constexpr int KK = K / 32;
  constexpr int kDepth = 3;  // steps whose operands are in flight
  // The state's three parts [v][k], double-buffered; keys in the images' order.
  __shared__ __align__(16) __bf16 sb[2][3][16 * K];
  const int lane = threadIdx.x & 63, wid = wave_index();
  const int l15 = lane & 15, lg = lane >> 4;
  const int nt = V / 16;
  // The column tiles of one head read the same transitions: on one XCD.
  const int64_t xcd = blockIdx.x & 7, r = blockIdx.x >> 3;
  const int v0 = static_cast<int>(r % nt) * 16;
  const int64_t item = (r / nt) * 8 + xcd;
  if (item >= p.N * p.HV) return;
  if (!*p.seg_len) return;
  const int hv = static_cast<int>(item % p.HV);
  const WaveSegs ws = wave_segs(p);
  const int nn = static_cast<int>(item / p.HV);
  const int seg0 = __builtin_amdgcn_readlane(ws.incl - ws.cnt, nn);
  const int cnt = min(__builtin_amdgcn_readlane(ws.cnt, nn), p.seg_max - seg0);
  if (cnt <= 1) return;  // no boundary
  const int64_t sh0 = static_cast<int64_t>(seg0) * p.HV + hv;
  if (v0 == 0 && wid == 0) {
    int over = 0;
    for (int i = lane; i < 2 * (cnt - 2); i += kWave)
      over |= p.seg_over[2 * (sh0 + (1 + (i >> 1)) * static_cast<int64_t>(p.HV)) + (i & 1)];
    const uint64_t any = __ballot(over != 0);
    if (lane == 0) p.seg_bad[item] = any != 0;
  }
  const int r4 = 16 * wid + 4 * lg;  // first of the lane's four state rows
  const int kpos = 32 * (wid >> 1) + 8 * lg + 4 * (wid & 1);  // their place in the images' order
  // Per-step strides and the lane's place in each, so that a step's
  // addresses are one scalar base plus one lane offset.
  float* bseg = p.seg_b + sh0 * K * V;
  const int64_t bstep = static_cast<int64_t>(p.HV) * K * V;
  const uint32_t boff = static_cast<uint32_t>(r4) * V + v0 + l15;
  const char* mseg = p.seg_m + sh0 * kSegImg + wid * (KK * 3072);
  const int64_t mstep = static_cast<int64_t>(p.HV) * kSegImg;
  struct Stage {
    bf8_t m[KK][3];
    f4_t b;
    float c;
  } st[kDepth];
  auto load_b = [&](int i) {
    const float* b = bseg + i * bstep;
    return f4_t{b[boff], b[boff + V], b[boff + 2 * V], b[boff + 3 * V]};
  };
  auto load = [&](Stage& t, int i) {
    t.c = p.seg_c[sh0 + static_cast<int64_t>(i) * p.HV];
    t.b = load_b(i);
    const char* m = mseg + i * mstep;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int u = 0; u < 3; ++u)
        t.m[kk][u] = *reinterpret_cast<const bf8_t*>(m + 3072 * kk + 1024 * u + 16u * lane);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto store = [&](int i, const f4_t& v) {
    float* out = bseg + i * bstep;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[boff + e * V] = v[e];
  };
  // Loads and stores count in one in-order counter, so a wait for a load
  // waits for everything issued before it: every load of the loop is
  // unconditional (past the last step it repeats that step's, unused), in
  // the order the steps take them, and a step stores the state it starts
  // from, ahead of its loads.
  const int last = cnt - 2;
  f4_t s = load_b(0);
  __builtin_amdgcn_sched_barrier(0);
  if (last > 0) {
#pragma unroll
    for (int u = 0; u < kDepth; ++u) load(st[u], min(u + 1, last));
  }
  auto step = [&](Stage& t, int i) {
    const int buf = i & 1;
    Vec<__bf16, 4> part[3];
    split4x3(s, part);
#pragma unroll
    for (int u = 0; u < 3; ++u)
      *reinterpret_cast<Vec<__bf16, 4>*>(&sb[buf][u][sb8_off(l15, kpos)]) = part[u];
    store(i - 1, s);
    // State copy complete; the other buffer's readers passed the barrier before.
    __syncthreads();
    // Parts h, m, l of each: every product but m l, l m and l l (2^-24).
    f4_t acc[3] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      bf8_t x[3];
#pragma unroll
      for (int u = 0; u < 3; ++u)
        x[u] = *reinterpret_cast<const bf8_t*>(&sb[buf][u][sb8_off(l15, 32 * kk + 8 * lg)]);
#pragma unroll
      for (int u = 0; u < 3; ++u)
#pragma unroll
        for (int w = 0; w + u < 3; ++w) acc[u + w] = mfma16(t.m[kk][w], x[u], acc[u + w]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = fmaf(t.c, s[e], t.b[e]) + (acc[0][e] + (acc[1][e] + acc[2][e]));
    __builtin_amdgcn_sched_barrier(0);
    load(t, min(i + kDepth, last));
  };
  int i = 1;
  for (; i + kDepth - 1 <= last; i += kDepth) {
#pragma unroll
    for (int u = 0; u < kDepth; ++u) step(st[u], i + u);
  }
#pragma unroll
  for (int u = 0; u < kDepth - 1; ++u)
    if (i + u <= last) step(st[u], i + u);
  if (last > 0) store(last, s);
}

template <int K, typename GT, typename BT>
int launch_chunk(const ChunkParams& p, int64_t V, hipStream_t s) {
  int st;
  if (p.N > kWaveSeqs) {  // else the kernels look chunks up themselves
    hipLaunchKernelGGL(chunk_offsets_kernel<ChunkParams>, dim3(1), dim3(256), 0, s, p,
                       p.seq_order, p.ctab, p.NTmax);
    if ((st = launch_status())) return st;
  }
  const int64_t prep_blocks = p.NTmax * ((p.HV + 3) / 4);
  if (prep_blocks >= INT32_MAX) return XK_ERR_UNSUPPORTED;
  hipLaunchKernelGGL((gdn_chunk_prep_kernel<K, GT, BT>),
                     dim3(static_cast<uint32_t>(prep_blocks) + (p.N <= kWaveSeqs ? 1 : 0)),
                     dim3(kTh), 0, s, p);
  st = launch_status();
  if (st) return st;
  const int64_t items = p.N * p.HV;
  if (V % 64 == 0 && p.seg_max > 0) {
    const int nvt = static_cast<int>(V / 64);
    const int64_t seg_items = cdiv(static_cast<int64_t>(p.seg_max) * p.HV, 8) * 8;
    const int64_t sum_items = cdiv((p.seg_max - p.N) * p.HV, 8) * 8;
    hipLaunchKernelGGL((gdn_chunk_state8_kernel<K, kSegSum>), dim3(sum_items * (nvt + K / 64)),
                       dim3(kTh8), 0, s, p, nvt);
    if ((st = launch_status())) return st;
    hipLaunchKernelGGL((gdn_chunk_combine_kernel<K>), dim3(cdiv(items, 8) * 8 * (V / 16)),
                       dim3(kTh8), 0, s, p, static_cast<int>(V));
    if ((st = launch_status())) return st;
    hipLaunchKernelGGL((gdn_chunk_state8_kernel<K, kSegOut>), dim3(seg_items * nvt), dim3(kTh8), 0,
                       s, p, nvt);
  } else if (V % 64 == 0) {
    const int nvt = static_cast<int>(V / 64);
    const int64_t blocks = cdiv(items, 8) * 8 * nvt;
    hipLaunchKernelGGL((gdn_chunk_state8_kernel<K, kSegNone>), dim3(blocks), dim3(kTh8), 0, s, p,
                       nvt);
  } else {
    constexpr int BV = 32;
    const int nvt = static_cast<int>(V / BV);
    const int64_t blocks = cdiv(items, 8) * 8 * nvt;
    hipLaunchKernelGGL((gdn_chunk_state_kernel<K, bf16, BV>), dim3(blocks), dim3(kTh), 0, s, p, nvt);
  }
  return launch_status();
}

// g and beta each come in fp32 or bf16 (chunk.py's callers pass fp32 g and
// bf16 beta).
template <int K, typename GT>
int chunk_beta(const ChunkParams& p, int64_t V, xk_dtype bdt, hipStream_t s) {
  if (bdt == XK_F32) return launch_chunk<K, GT, float>(p, V, s);
  if (bdt == XK_BF16) return launch_chunk<K, GT, bf16>(p, V, s);
  return XK_ERR_UNSUPPORTED;
}

int64_t nt_max(int64_t total_tokens, int64_t N) { return total_tokens / kC + N; }

// Whether a call takes the segmented state pass, and its workspace past the
// records.  The lengths are not known here.  Several sequences are taken to
// be equally long, where segments gain least: with the same tokens a longer
// sequence lengthens the chain in order and leaves the segments' work as it
// is, so a batch that is offered the passes always takes them.  (Two idle
// passes cost 3 to 4 us, 3% of 4 equal sequences of 2,048 tokens x 16
// v-heads, more than it is right to take from batches that cannot gain.)
constexpr int64_t kSegHead = 256;  // the plan's word; always part of the size
struct SegPlan {
  int segs = 0;  // most segments; 0: whole sequences
  int64_t bytes = kSegHead;
};
SegPlan seg_plan(int64_t total_tokens, int64_t N, int64_t HV, int64_t K, int64_t V, int cus) {
  SegPlan r;
  const int64_t tiles = HV * (V / 64);
  if (N <= 0 || N > kSegSeqs || V % 64 != 0 || N * tiles > cus) return r;
  const int64_t longest = std::max<int64_t>(cdiv(cdiv(total_tokens, N), kC), 1);
  auto cost = [&](int s, int64_t len, int64_t sums, int64_t outs) {
    return seg_cost(s, static_cast<int>(len), static_cast<int>(sums),
                    static_cast<int>(sums - N * 2 * HV), static_cast<int>(outs), cus);
  };
  // (At least 2 us must be gained: the model is good to a few percent.)
  float best = cost(1, longest, 0, N * tiles) - 2.f;
  // The smallest s of every length, while s segments of one chunk could gain:
  // every call pays for this loop (63 candidates per width took 0.3 us).
  for (int64_t s = 2; s <= 64 && 25.f + 1.4f * (s - 2) < best;) {
    const int64_t len = cdiv(longest, s), segs = N * cdiv(longest, len);
    const float c =
        cost(static_cast<int>(s), len, (segs - N) * (tiles + 2 * HV), segs * tiles);
    if (c < best) {
      best = c;
      r.segs = static_cast<int>(segs);
    }
    if (len <= 1) break;
    s = cdiv(longest, len - 1);
  }
  // Several sequences: room for one round of kSegOut blocks.
  if (r.segs && N > 1) r.segs = static_cast<int>(std::max<int64_t>(r.segs, cus / tiles) + N / 2);
  if (r.segs)
    r.bytes = kSegHead + align256(4 * N * HV) + align256(8 * r.segs * HV) + align256(4 * r.segs * HV) +
              r.segs * HV * (kSegImg + K * V * 4);
  return r;
}

}  // namespace
}  // namespace xk

using namespace xk;

namespace {

// Widest states that the size makes room for; wider ones run in order.
constexpr int64_t kSegMaxV = 256;

// The least a call runs in (without segments).
int64_t least_workspace(int64_t total_tokens, int64_t N, int64_t HV) {
  const int64_t nt = nt_max(total_tokens, N);
  return align256(4 * (N + 1)) + align256(4 * N) + align256(8 * nt) + kDump + nt * HV * kRec;
}

}  // namespace

extern "C" int64_t xk_gdn_chunk_workspace_bytes(int64_t total_tokens, int64_t num_seqs,
                                                int64_t HV) {
  if (total_tokens < 0 || num_seqs < 0 || HV <= 0) return -1;
  // V is not known here: room for the segments of any up to kSegMaxV.
  int64_t seg = 0;
  const int cus = num_cus();
  for (int64_t V = 64; V <= kSegMaxV; V += 64)
    seg = std::max(seg, seg_plan(total_tokens, num_seqs, HV, 128, V, cus).bytes);
  return least_workspace(total_tokens, num_seqs, HV) + seg;
}

namespace xk {
namespace {

// Argument checks shared by xk_gdn_chunk_fwd and xk_gdn_chunk_fwd_noalloc
// (everything but the workspace).  *empty is set for a call with no work
// (N or total_tokens 0), which returns XK_OK before its pointers are
// checked.
int chunk_args_status(const void* q, const void* k, const void* v, xk_dtype dtype,
                      const void* g, xk_dtype g_dtype, const void* beta, xk_dtype beta_dtype,
                      const void* o, const void* cu_seqlens, xk_dtype cu_dtype, int64_t N,
                      int64_t total_tokens, int64_t H, int64_t HV, int64_t K, int64_t V,
                      int64_t sqk, int64_t sv, bool* empty) {
  *empty = false;
  if (N < 0 || total_tokens < 0 || H <= 0 || HV <= 0 || HV % H != 0)
    return XK_ERR_INVALID;
  // bf16 only, as the reference entry point (q/k feed the bf16 MFMA as-is).
  if (dtype != XK_BF16) return XK_ERR_UNSUPPORTED;
  if (g_dtype != XK_F32 && g_dtype != XK_BF16) return XK_ERR_UNSUPPORTED;
  if (beta_dtype != XK_F32 && beta_dtype != XK_BF16) return XK_ERR_UNSUPPORTED;
  if (cu_dtype != XK_I32 && cu_dtype != XK_I64) return XK_ERR_UNSUPPORTED;
  if (K != 128 || V % 32 != 0 || V <= 0) return XK_ERR_UNSUPPORTED;
  // Row pitches of q / k and v / o in bytes feed 24-bit multiplies.
  if (H * K * 2 >= (int64_t{1} << 24) || HV * V * 2 >= (int64_t{1} << 24) ||
      sqk * 2 >= (int64_t{1} << 24) || sv * 2 >= (int64_t{1} << 24))
    return XK_ERR_UNSUPPORTED;
  // Rows must not overlap and start at 16-byte boundaries.
  if (sqk < H * K || sv < HV * V || sqk % 8 != 0 || sv % 8 != 0) return XK_ERR_INVALID;
  if (N == 0 || total_tokens == 0) {
    *empty = true;
    return XK_OK;
  }
  // Token indices travel as int32 in the chunk table.
  if (total_tokens > INT32_MAX - kC) return XK_ERR_UNSUPPORTED;
  if (!q || !k || !v || !g || !beta || !o || !cu_seqlens) return XK_ERR_INVALID;
  if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) || !aligned(o, 8))
    return XK_ERR_INVALID;
  return XK_OK;
}

}  // namespace
}  // namespace xk

extern "C" int xk_gdn_chunk_fwd_strided(
    const void* q, const void* k, int64_t stride_qk_tok, const void* v, int64_t stride_v_tok,
    xk_dtype dtype, const void* g, xk_dtype g_dtype, const void* beta, xk_dtype beta_dtype, void* o,
    const float* initial_state, float* final_state, const void* cu_seqlens,
    xk_dtype cu_dtype, int64_t N, int64_t total_tokens, int64_t H, int64_t HV,
    int64_t K, int64_t V, float scale, int use_qk_l2norm, void* workspace,
    size_t workspace_bytes, void* stream) {
  bool empty = false;
  const int ast =
      chunk_args_status(q, k, v, dtype, g, g_dtype, beta, beta_dtype, o, cu_seqlens, cu_dtype, N,
                        total_tokens, H, HV, K, V, stride_qk_tok, stride_v_tok, &empty);
  if (ast != XK_OK || empty) return ast;
  const int64_t need = least_workspace(total_tokens, N, HV);
  if (!workspace || static_cast<int64_t>(workspace_bytes) < need) return XK_ERR_WORKSPACE;
  if (!aligned(workspace, 256)) return XK_ERR_WORKSPACE;
  ChunkParams p{};
  p.q = q;
  p.k = k;
  p.v = v;
  p.sqk = static_cast<uint32_t>(stride_qk_tok);
  p.sv = static_cast<uint32_t>(stride_v_tok);
  p.g = g;
  p.beta = beta;
  p.o = o;
  p.h0 = initial_state;
  p.ht = final_state;
  p.cu = cu_seqlens;
  p.cu_i64 = cu_dtype == XK_I64;
  char* ws = static_cast<char*>(workspace);
  // 16 N <= align256(4 (N + 1)) + align256(4 N) + align256(8 N) for every N
  // up to kWaveSeqs.
  p.seqtab = reinterpret_cast<int4*>(ws);
  p.chunk_off = reinterpret_cast<int32_t*>(ws);
  ws += align256(4 * (N + 1));
  p.seq_order = reinterpret_cast<int32_t*>(ws);
  ws += align256(4 * N);
  p.ctab = reinterpret_cast<int2*>(ws);
  ws += align256(8 * nt_max(total_tokens, N));
  p.dump = reinterpret_cast<bf16*>(ws);
  p.rec = ws + kDump;
  p.N = N;
  p.NTmax = nt_max(total_tokens, N);
  p.T = total_tokens;
  p.H = static_cast<int>(H);
  p.HV = static_cast<int>(HV);
  p.scale = scale;
  p.l2norm = use_qk_l2norm;
  // Segments of a sequence run side by side, the first from the initial state
  // while the last writes the final state: where the two overlap (a state
  // updated in place), whole sequences run, whose blocks each read their part
  // of the state before they write it.
  const uintptr_t s0 = reinterpret_cast<uintptr_t>(initial_state),
                  s1 = reinterpret_cast<uintptr_t>(final_state);
  const uintptr_t state_bytes = static_cast<uintptr_t>(N * HV * K * V) * 4;
  const bool in_place = s0 && s1 && s0 < s1 + state_bytes && s1 < s0 + state_bytes;
  const SegPlan plan = in_place || V > kSegMaxV
                           ? SegPlan{}
                           : seg_plan(total_tokens, N, HV, K, V, num_cus());
  if (plan.segs && static_cast<int64_t>(workspace_bytes) >=
                       xk_gdn_chunk_workspace_bytes(total_tokens, N, HV)) {
    char* seg = p.rec + p.NTmax * HV * kRec;
    p.seg_max = plan.segs;
    p.seg_cus = num_cus();
    p.seg_nvt = static_cast<int>(V / 64);
    p.seg_len = reinterpret_cast<int32_t*>(seg);
    seg += kSegHead;
    p.seg_bad = reinterpret_cast<int32_t*>(seg);
    seg += align256(4 * N * HV);
    p.seg_over = reinterpret_cast<int32_t*>(seg);
    seg += align256(8 * plan.segs * HV);
    p.seg_c = reinterpret_cast<float*>(seg);
    seg += align256(4 * plan.segs * HV);
    p.seg_m = seg;
    p.seg_b = reinterpret_cast<float*>(seg + plan.segs * HV * kSegImg);
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (g_dtype == XK_F32) return chunk_beta<128, float>(p, V, beta_dtype, s);
  return chunk_beta<128, bf16>(p, V, beta_dtype, s);
}

extern "C" int xk_gdn_chunk_fwd(
    const void* q, const void* k, const void* v, xk_dtype dtype, const void* g,
    xk_dtype g_dtype, const void* beta, xk_dtype beta_dtype, void* o,
    const float* initial_state, float* final_state, const void* cu_seqlens,
    xk_dtype cu_dtype, int64_t N, int64_t total_tokens, int64_t H, int64_t HV,
    int64_t K, int64_t V, float scale, int use_qk_l2norm, void* workspace,
    size_t workspace_bytes, void* stream) {
  return xk_gdn_chunk_fwd_strided(q, k, H * K, v, HV * V, dtype, g, g_dtype, beta, beta_dtype, o,
                                  initial_state, final_state, cu_seqlens, cu_dtype, N,
                                  total_tokens, H, HV, K, V, scale, use_qk_l2norm, workspace,
                                  workspace_bytes, stream);
}

// ---------------------------------------------------------------------------
// xk_gdn_chunk_fwd_noalloc: the same pipeline with its workspace in a static
// device buffer.  Each GPU holds its own copy of `scratch` from the moment
// this code object is loaded on it until the process ends.  In host code the
// name `scratch` is only a handle for the runtime: the device address of a
// GPU's copy comes from hipGetSymbolAddress, called once per device with that
// device current, and only that address is handed to the kernels.  Every call
// rewrites the parts of the workspace it reads (chunk table, offsets,
// records) before reading them, so nothing needs clearing between calls.
// ---------------------------------------------------------------------------
namespace {

constexpr int64_t kNoAllocScratchBytes = int64_t{64} << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_addr[kMaxDevices];
std::mutex g_scratch_mu;

// Device address of the current device's `scratch` (looked up on the first
// call per device).  `stream` must belong to the current device.
int scratch_on_current_device(hipStream_t stream, void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return static_cast<int>(e);
  if (dev < 0 || dev >= kMaxDevices) return XK_ERR_UNSUPPORTED;
  hipDevice_t sdev = -1;
  e = hipStreamGetDevice(stream, &sdev);
  if (e != hipSuccess) return static_cast<int>(e);
  if (sdev != dev) return XK_ERR_INVALID;
  void* addr = g_scratch_addr[dev].load(std::memory_order_acquire);
  if (!addr) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    addr = g_scratch_addr[dev].load(std::memory_order_relaxed);
    if (!addr) {
      e = hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch));
      if (e != hipSuccess) return static_cast<int>(e);
      if (!addr) return XK_ERR_UNSUPPORTED;
      g_scratch_addr[dev].store(addr, std::memory_order_release);
    }
  }
  *out = addr;
  return XK_OK;
}

}  // namespace

extern "C" int xk_gdn_chunk_fwd_noalloc(
    const void* q, const void* k, const void* v, xk_dtype dtype, const void* g,
    xk_dtype g_dtype, const void* beta, xk_dtype beta_dtype, void* o,
    const float* initial_state, float* final_state, const void* cu_seqlens,
    xk_dtype cu_dtype, int64_t N, int64_t total_tokens, int64_t H, int64_t HV,
    int64_t K, int64_t V, float scale, int use_qk_l2norm, void* stream) {
  // The same argument checks as xk_gdn_chunk_fwd, before the size check.
  bool empty = false;
  const int ast = chunk_args_status(q, k, v, dtype, g, g_dtype, beta, beta_dtype, o, cu_seqlens,
                                    cu_dtype, N, total_tokens, H, HV, K, V, H * K, HV * V, &empty);
  if (ast != XK_OK || empty) return ast;
  const int64_t need = least_workspace(total_tokens, N, HV);
  if (need > kNoAllocScratchBytes) return XK_ERR_SCRATCH;
  void* ws = nullptr;
  const int st = scratch_on_current_device(static_cast<hipStream_t>(stream), &ws);
  if (st != XK_OK) return st;
  return xk_gdn_chunk_fwd(q, k, v, dtype, g, g_dtype, beta, beta_dtype, o, initial_state,
                          final_state, cu_seqlens, cu_dtype, N, total_tokens, H, HV, K, V,
                          scale, use_qk_l2norm, ws, static_cast<size_t>(kNoAllocScratchBytes),
                          stream);
}
