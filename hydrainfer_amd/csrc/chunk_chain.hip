// chunk_chain.hip — recurrences over portions of prompts, sixteen tokens at a time (chunk_scan.hip says how), in two launches: what
// does not depend on the state — A, M, prefixed queries, suffixed keys, all of it vector work and a serial substitution — is made for all
// chunks at once on the whole chip, and the chain of chunks is left with the products of the state.  One launch has these made beside
// the chain, on the same SIMDs and once per 64 value channels.  Few long chains go in segments, in a launch more (segment_chunks).
// What bounds the chain: a chunk is 104 float products a wave under the delta rule with 128 x 128 (68 without write strengths), 32 cycles
// each, where a wave holds all keys of 16 value channels, and 140 (100) vector instructions that do not run beside the products of
// their own wave (a multiplication behind a product costs 7 cycles; those of other waves cost it nothing).  So the keys of 16 value channels are
// dealt to two waves, or to four where workgroups are few: a chunk then takes 1.1 to 1.7 us instead of 2.0 to 2.7 (reads from LDS
// behind the barrier 0.3, products 0.25 a product with the state, sums and results 0.2, barrier 0.1).  Results and, under the delta rule, what the keys
// read from the old state are shares of the parts; results leave by the waves that bring rows in, which add the shares up in
// double.  A share comes in two numbers, what the state gave and what the chunk gave, so that it is rounded no more often than the
// whole was: 2-norm of the error against 64 bits, one launch and two, 3 portions of 200 - 600 tokens, 16 heads of 128 x 128: delta 1.08
// 1.02, decay 0.85 0.77, bonus 0.82 0.79 e-7 (added up in float and in one number 1.09, 0.85, 0.87).
// Measured, one launch and two, us: 4 portions of 1000 tokens, 8 heads of 128 x 128: delta rule 166 and 131, decayed sum 127 and 83,
// gated form (with its norm) 173 and 87, bonus form 160 and 101; one of 1151, 32 heads: 188 150, 144 95, 197 96, 182 113; 64 x 64: decayed sum 92 86, gated
// form 121 81, bonus form 109 103; delta rule 122 128, which stays with one launch.  4 portions of 797 - 1151 tokens, 32 heads of 128 x 128, gated form 206 and 171 (53 of them the
// first launch, 560 vector instructions a wave of four tokens and 164 MB written; delta rule 190 and 235, so the first launch is weighed
// against the chain, chunk_scan_workspace).
#include "chunk_parts.h"
#include <algorithm>
#include <cmath>

namespace {

// The chunks of a launch, wherever they lie: chunk c of sequence s has number q_cu[s] / 16 + s + c (some numbers are nobody's).
struct ChunkAt {
  int64_t t0;               // its first token
  int n;                    // tokens; 0: nobody's
};
__device__ __forceinline__ int64_t chunk_number(int64_t t_begin, int seq) { return t_begin / C + seq; }
__device__ __forceinline__ ChunkAt chunk_at(const ChunkScanArgs& a, int64_t number) {
  const int lane = threadIdx.x & 63;
  int seq = -1;
  for (int s0 = 0; s0 < a.n_seq; s0 += 64) {              // the last sequence that starts at or before this number
    const int s = s0 + lane;
    const int here = __popcll(__builtin_amdgcn_ballot_w64(s < a.n_seq && chunk_number(a.q_cu[min(s, a.n_seq - 1)], s) <= number));
    seq += here;
    if (here < 64) break;
  }
  if (seq < 0) return ChunkAt{0, 0};
  const int64_t t_begin = a.q_cu[seq], n_tok = a.q_cu[seq + 1] - t_begin, first = (number - chunk_number(t_begin, seq)) * C;
  return ChunkAt{t_begin + first, (int)(first < n_tok ? (n_tok - first < C ? n_tok - first : C) : 0)};
}

// N floats on their way to LDS: NT threads
template <int N, int NT>
struct MadeRows {
  static constexpr int P = (N / 4 + NT - 1) / NT;
  f32x4 p[P];
  __device__ __forceinline__ void fetch(const float* from, int tid) {
#pragma unroll
    for (int i = 0; i < P; ++i) p[i] = *reinterpret_cast<const f32x4*>(from + 4 * min(tid + i * NT, N / 4 - 1));
  }
  __device__ __forceinline__ void store(float* lds, int tid) const {
#pragma unroll
    for (int i = 0; i < P; ++i)
      if (tid + i * NT < N / 4) *reinterpret_cast<f32x4*>(lds + 4 * (tid + i * NT)) = p[i];
  }
};

// ---------------------------------------------------------------------------------------------------------------
// What does not depend on the state, all chunks at once.
// ---------------------------------------------------------------------------------------------------------------
// What one chunk needs besides its rows: A | M (T while it is made; delta rule) | prefix, suffix, what the prefix's rounding left over
template <bool DELTA>
constexpr int kMadeHead = (DELTA ? 2 : 1) * C * RA + 3 * C;

// A wave's (x k^T)[i, j] with rows i = 4 g + e and column j = m: tokens 4 e + g and t_m; N chains
template <int KP, int N>
__device__ __forceinline__ f32x4 with_keys(const float* rows_x, const float* k, int m, int g) {
  constexpr int RS = KP + 4;
  f32x4 p[N];
#pragma unroll
  for (int i = 0; i < N; ++i) p[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kt = 0; kt < KP / 16; ++kt) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(rows_x + m * RS + 16 * kt + 4 * g);
    const f32x4 y = *reinterpret_cast<const f32x4*>(k + m * RS + 16 * kt + 4 * g);
#pragma unroll
    for (int e = 0; e < 4; ++e) p[(4 * kt + e) % N] = mma4(x[e], y[e], p[(4 * kt + e) % N]);
  }
#pragma unroll
  for (int n = N / 2; n > 0; n >>= 1)
#pragma unroll
    for (int i = 0; i < n; ++i) p[i] += p[i + n];
  return p[0];
}
__device__ __forceinline__ void chunk_decays(const float* sc, float (&d)[C]) {
#pragma unroll
  for (int i = 0; i < C / 4; ++i) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(sc + 4 * i);
#pragma unroll
    for (int e = 0; e < 4; ++e) d[4 * i + e] = x[e];
  }
}
// A, prefixes and suffixes: with sixteen chains and products of decays rounded once, as A's rounding is the larger part of a
// result's error.  scalars: the chunk's per head numbers besides.
template <int KP>
__device__ __forceinline__ void make_A(const float* q, const float* k, const float* sc, float* A, float* scalars, int m, int g, int t_m) {
  const f32x4 xk = with_keys<KP, 16>(q, k, m, g);
  float d[C];
  chunk_decays(sc, d);
  Product run, mine[4];                                   // run = prod(t_m < r <= t) d_r, kept at the lane's four rows
#pragma unroll
  for (int t = 0; t < C; ++t) {
    run.by(t > t_m ? d[t] : 1.f);
    const bool here = (t & 3) == 0 || (t & 3) == g;
    mine[t >> 2].hi = here ? run.hi : mine[t >> 2].hi;
    mine[t >> 2].lo = here ? run.lo : mine[t >> 2].lo;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) A[(4 * g + e) * RA + m] = t_m <= 4 * e + g ? mine[e].times(xk[e]) : 0.f;
  if (g == 0) scalars[C + m] = run.value();               // behind token t_m
  if (m == 0) {                                           // up to the rows' tokens: the first one's decay and all behind it
    f32x4 prefix, rest;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      prefix[e] = mine[e].times(d[0]);
      rest[e] = mine[e].rest(d[0], prefix[e]);
    }
    *reinterpret_cast<f32x4*>(scalars + 4 * g) = prefix;
    *reinterpret_cast<f32x4*>(scalars + 2 * C + 4 * g) = rest;
  }
}
template <int KP>
__device__ __forceinline__ void make_M(const float* k, const float* sc, float* A, int m, int g, int t_m) {      // A: T (by tokens), then M
  const f32x4 xk = with_keys<KP, 4>(k, k, m, g);
  float d[C], run = 1.f, mine[4];
  chunk_decays(sc, d);
#pragma unroll
  for (int t = 0; t < C; ++t) {
    run = t > t_m ? run * d[t] : 1.f;
    mine[t >> 2] = (t & 3) == 0 || (t & 3) == g ? run : mine[t >> 2];
  }
  const f32x4 b = *reinterpret_cast<const f32x4*>(sc + 2 * C + 4 * g);
#pragma unroll
  for (int e = 0; e < 4; ++e) A[(4 * e + g) * RA + t_m] = t_m < 4 * e + g ? b[e] * xk[e] * mine[e] : 0.f;      // (T: by tokens)
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // column t_m of (I + T)^-1: x_t = [t == t_m] - sum(s < t) T[t, s] x_s
  float x[C];
#pragma unroll
  for (int t = 0; t < C; ++t) {
    float s0 = t == t_m ? 1.f : 0.f, s1 = 0.f;
#pragma unroll
    for (int s = 0; s < t; s += 4) {
      const f32x4 T = *reinterpret_cast<const f32x4*>(A + t * RA + s);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (s + e >= t) continue;
        if (e & 1) s1 -= T[e] * x[s + e];
        else s0 -= T[e] * x[s + e];
      }
    }
    x[t] = s0 + s1;
    if (t & 1) asm volatile("" ::: "memory");           // (two rows of T in registers at a time, not all of them)
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();                      // T has been read
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (g == 0) {
#pragma unroll
    for (int t = 0; t < C; ++t) A[row_of_token(t) * RA + m] = x[t];
  }
}

// One decay per token and head: wave 0 A, prefixes and suffixes, wave 1 M.  (As chunk_head_kernel makes them; made by calls of these
// functions there, its chunks take 6 % longer.)
template <int KP, bool DELTA, typename QK, bool VEC>
__global__ __launch_bounds__(128, 4) void chunk_head_make_kernel(ChunkScanArgs a) {
  constexpr int RS = KP + 4, kMade = kMadeHead<DELTA>;
  __shared__ __attribute__((aligned(16))) float rows[2 * C * RS + 3 * C + kMade];
  const int head = blockIdx.x % (unsigned)a.heads;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, m = lane & 15;
  const ChunkAt at = chunk_at(a, blockIdx.x / (unsigned)a.heads);
  if (at.n <= 0) return;                                  // (the whole workgroup)
  const int qk_head = head / (a.heads / a.qk_heads);
  float *sc = rows + 2 * C * RS, *A = sc + 3 * C;
  Rows<QK, VEC, KP, 64> x;
  const int64_t stride = wave == 0 ? a.q_stride : a.k_stride;
  x.fetch((const typename QK::storage*)(wave == 0 ? a.q : a.k) + at.t0 * stride + (int64_t)qk_head * a.K, stride, 0, a.K, at.n, lane);
  const int64_t th = (at.t0 + min(m, at.n - 1)) * a.heads + head;
  const float decay = a.decay[th], beta = DELTA ? a.beta[th] : 0.f;
  x.store(rows + wave * C * RS, 0, a.K, at.n, 1.f, lane);
  if (threadIdx.x < C) {                                  // (decays by token, the others by row; a row past the portion changes nothing)
    sc[m] = m < at.n ? decay : 1.f;
    sc[2 * C + row_of_token(m)] = m < at.n ? beta : 0.f;
  }
  lds_barrier();
  if (wave == 0) make_A<KP>(rows, rows + C * RS, sc, A, A + kMade - 3 * C, m, g, row_of_token(m));
  else if constexpr (DELTA) make_M<KP>(rows + C * RS, sc, A + C * RA, m, g, row_of_token(m));
  lds_barrier();
  float* to = a.made + (int64_t)blockIdx.x * kMade;
  for (int i = 4 * threadIdx.x; i < kMade; i += 4 * 128) *reinterpret_cast<f32x4*>(to + i) = *reinterpret_cast<const f32x4*>(A + i);
}

// One decay per token and key channel.
template <int KP, int FORM, typename QK, bool VEC>
__global__ __launch_bounds__(256, 4) void chunk_channel_make_kernel(ChunkScanArgs a) {
  constexpr int RS = KP + 4, NP = KP / 64, kGate = kGateFloats<KP, FORM>, kMade = kMadeChannel<KP, FORM>;
  __shared__ __attribute__((aligned(16))) float lds[kGate + kMade];
  const int head = blockIdx.x % (unsigned)a.heads;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, d0 = NP * lane;
  const ChunkAt at = chunk_at(a, blockIdx.x / (unsigned)a.heads);
  if (at.n <= 0) return;                                  // (the whole workgroup)
  const int qk_head = head / (a.heads / a.qk_heads);
  const ChannelBias<NP, FORM> own(a, head, d0);
  const int64_t d_stride = (int64_t)a.heads * a.K;
  GateRows<KP, FORM, QK, VEC> x;
  x.fetch((const typename QK::storage*)a.q + at.t0 * a.q_stride + (int64_t)qk_head * a.K, a.q_stride, (const typename QK::storage*)a.k + at.t0 * a.k_stride + (int64_t)qk_head * a.K,
          a.k_stride, FORM == hxm::kChunkGated ? nullptr : a.decay + at.t0 * d_stride + (int64_t)head * a.K, d_stride, at.n, a.K, wave, d0);
  float* P = lds + kGate;
  for (int i = threadIdx.x; i < C * RA; i += 256) P[C * RS + KP * RA + i] = 0.f;      // (above A's diagonal)
  x.store(lds, own, at.n, a.K, wave, d0);
  lds_barrier();
  finish_chunk<KP, FORM>(lds, P, own, place_in_A(wave, lane), wave, lane);
  lds_barrier();
  float* to = a.made + (int64_t)blockIdx.x * kMade;
  for (int i = 4 * threadIdx.x; i < kMade; i += 4 * 256) *reinterpret_cast<f32x4*>(to + i) = *reinterpret_cast<const f32x4*>(P + i);
}

// ---------------------------------------------------------------------------------------------------------------
// The chain.  Eight consumer waves hold the state, 32 key channels of 16 value channels each; four more bring in what a chunk takes,
// kAhead chunks ahead of the interval that puts it in LDS, and take results out.
// ---------------------------------------------------------------------------------------------------------------
// delta rule: q | k | v | write strength, and A | M | scalars; decayed sum: the same with value scales and without M; a decay per
// channel: v, and what chunk_channel_make_kernel makes
template <int KP, int FORM, bool CHANNEL, int KS>
struct Image {
  static constexpr int W = 16 * 8 / KS, WS = W + 4;       // value channels a workgroup
  static constexpr bool DELTA = FORM == hxm::kChunkDelta;
  static constexpr int kMade = CHANNEL ? kMadeChannel<KP, CHANNEL ? FORM : hxm::kChunkDecay> : kMadeHead<DELTA>;
  static constexpr int kRows = CHANNEL ? 0 : 2 * C * (KP + 4) + C;
  static constexpr int kFloats = kMade + kRows + C * WS;
  static constexpr int kImages = DELTA ? 3 : 2;
  static constexpr int kShares = KS * C * WS;             // the key parts' shares of y, or of a chunk's results
  // results whose rounding shows (the gated form's are rounded to an activation behind its norm) in two numbers
  static constexpr int kResult = (FORM == hxm::kChunkGated ? 1 : 2) * kShares;
  static constexpr int kLds = kImages * kFloats + 2 * kResult + (DELTA ? 2 * kShares : 0);
};

// Few chains leave most compute units idle, and a chain is as long as its portion.  The state behind a segment of a portion is what its
// own tokens give from an empty state and what its decays leave of the state ahead of it, so the segments' states are made all at
// once by a launch ahead (kSegmentStates: the chain without queries and results), and the segments of every portion are then chains of
// their own (kSegmentResults), which put the state that they start from together out of those.
// Segment p of sequence s, `segment` chunks each, has number q_cu[s] / (16 segment) + s + p and, for every head, K V + 2 K floats in
// `segments`: the state behind the segment ahead of it (the first one's from the portion's true start, the others' from nothing; of
// segment 0 the start itself: the last segment may store the final state before the first one begins), and its product of decays, in
// double for the range.
enum { kWhole, kSegmentStates, kSegmentResults };
__host__ __device__ inline int64_t segment_state(const ChunkScanArgs& a) { return ((int64_t)a.K * a.V + 1) / 2 * 2; }      // (doubles behind it)
__device__ __forceinline__ float* segment_at(const ChunkScanArgs& a, int64_t number, int head) {
  return a.segments + (number * a.heads + head) * (int64_t)(segment_state(a) + 2 * a.K);
}
struct SegmentAt {
  int seq, p;               // seq < 0: nobody's
};
__device__ __forceinline__ SegmentAt segment_of(const ChunkScanArgs& a, int64_t number) {
  const int lane = threadIdx.x & 63, tokens = C * a.segment;
  int seq = -1;
  for (int s0 = 0; s0 < a.n_seq; s0 += 64) {              // the last sequence that starts at or before this number
    const int s = s0 + lane;
    const int here = __popcll(__builtin_amdgcn_ballot_w64(s < a.n_seq && a.q_cu[min(s, a.n_seq - 1)] / tokens + s <= number));
    seq += here;
    if (here < 64) break;
  }
  return seq < 0 ? SegmentAt{-1, 0} : SegmentAt{seq, (int)(number - (a.q_cu[seq] / tokens + seq))};
}
// what a product of decays becomes with one more: it does not leave the range while its factors are in theirs (what it leaves of an infinity is one)
__device__ __forceinline__ double decayed(double product, float d) {
  const double x = product * (double)d;
  return d != 0.f && fabs(x) < 1e-300 ? copysign(1e-300, x) : x;
}

template <int KP, int FORM, bool CHANNEL, int KS, typename QK, typename VT, bool VEC, int PASS>
__global__ __launch_bounds__(768) void chunk_chain_kernel(ChunkScanArgs a) {
  typedef Image<KP, FORM, CHANNEL, KS> I;
  constexpr int RS = KP + 4, KT = KP / 16 / KS, W = I::W, WS = I::WS, kMade = I::kMade, kLead = I::kImages - 2;
  constexpr bool DELTA = I::DELTA, BONUS = FORM == hxm::kChunkBonus;
  extern __shared__ __attribute__((aligned(16))) float lds[];      // images | results[2] | y[2]
  constexpr bool kResults = PASS != kSegmentStates;
  constexpr int kSkip = CHANNEL && !kResults ? C * RS : 0;      // (the queries)
  const int head = blockIdx.x, col0 = (int)blockIdx.y * W;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, m = lane & 15;
  int seq = blockIdx.z, part_at = 0;                      // part_at: the segment
  if constexpr (PASS != kWhole) {
    const SegmentAt at = segment_of(a, blockIdx.z);
    if (at.seq < 0) return;                               // (the whole workgroup, as below)
    seq = __builtin_amdgcn_readfirstlane(at.seq);
    part_at = __builtin_amdgcn_readfirstlane(at.p);
  }
  const int64_t t_seq = a.q_cu[seq], t_begin = PASS == kWhole ? t_seq : t_seq + (int64_t)part_at * a.segment * C;
  int n_tok = (int)(a.q_cu[seq + 1] - t_begin);
  if (n_tok <= 0) return;                                 // (the whole workgroup)
  bool last = true;
  if constexpr (PASS != kWhole) {
    last = n_tok <= a.segment * C;
    if (PASS == kSegmentStates && last) return;
    n_tok = min(n_tok, a.segment * C);
  }
  const int n_chunks = (n_tok + C - 1) / C;
  auto made = [&](int chunk) { return lds + chunk % I::kImages * I::kFloats; };
  auto rows = [&](int chunk) { return made(chunk) + kMade; };
  auto vals = [&](int chunk) { return made(chunk) + kMade + I::kRows; };
  auto outs = [&](int chunk) { return lds + I::kImages * I::kFloats + (chunk & 1) * I::kResult; };
  auto ys = [&](int chunk) { return lds + I::kImages * I::kFloats + 2 * I::kResult + (chunk & 1) * I::kShares; };      // (delta rule)
  auto rows_of = [&](int chunk) { return min(C, n_tok - chunk * C); };

  if (wave >= 4) {
    const int part = (wave - 4) % KS, cw = (wave - 4) / KS, col = col0 + 16 * cw + m, k0 = 16 * KT * part;
    float* slot = a.state + (int64_t)a.slots[seq] * a.slot_stride + (int64_t)head * a.K * a.V + (int64_t)k0 * a.V;
    State<KT> st;
    const bool fresh = a.positions[t_seq] == 0;
    double left[CHANNEL ? KT : 1][4];                     // (kSegmentStates: this segment's product of decays)
    if constexpr (PASS == kWhole) {
      st.load(slot, a.K - k0, a.V, col, g, fresh);
    } else if constexpr (PASS == kSegmentStates) {
      st.load(slot, a.K - k0, a.V, col, g, fresh || part_at > 0);
      if (part_at == 0) st.store(segment_at(a, blockIdx.z, head) + (int64_t)k0 * a.V, a.K - k0, a.V, col, g);
#pragma unroll
      for (int kt = 0; kt < (CHANNEL ? KT : 1); ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e) left[kt][e] = 1.0;
    } else if (part_at == 0) {
      const bool alone = last;                            // (nobody else reads or writes the slot's columns)
      st.load(alone ? slot : segment_at(a, blockIdx.z, head) + (int64_t)k0 * a.V, a.K - k0, a.V, col, g, alone && fresh);
    } else {
      const int64_t first = (int64_t)blockIdx.z - part_at;
      st.load(segment_at(a, first + 1, head) + (int64_t)k0 * a.V, a.K - k0, a.V, col, g, false);
#pragma unroll 1
      for (int p = 1; p < part_at; ++p) {                 // what segment p makes of the state behind the one ahead of it
        State<KT> own;
        own.load(segment_at(a, first + p + 1, head) + (int64_t)k0 * a.V, a.K - k0, a.V, col, g, false);
        const double* decays = reinterpret_cast<const double*>(segment_at(a, first + p, head) + segment_state(a));
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int kk = k0 + 16 * kt + 4 * g + e;
            st.S[kt][e] = (float)__builtin_fma(decays[min(kk, a.K - 1)], (double)st.S[kt][e], (double)own.S[kt][e]);
          }
      }
    }
    const int share = part * C * WS + 4 * g * WS + 16 * cw + m;      // this lane's column of rows 4 g ..
    // the keys' part of rows (token m) of x times the state; four chains of at most sixteen keys
    auto times_state = [&](const float* row) __attribute__((always_inline)) {
      f32x4 x[KT], o[4];
      read_row(x, row + k0);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = mma4(x[0][e], st.S[0][e], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int kt = 1; kt < KT; ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = mma4(x[kt][e], st.S[kt][e], o[e]);
      return (o[0] + o[1]) + (o[2] + o[3]);
    };
    auto put = [&](float* to, f32x4 v) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < 4; ++e) to[share + e * WS] = v[e];
    };
    if constexpr (DELTA) {
      lds_barrier();
      put(ys(0), times_state(rows(0) + C * RS + m * RS + 4 * g));
    }
    for (int c = 0; c < n_chunks; ++c) {
      lds_barrier();
      const float *p = made(c), *A = CHANNEL ? p + C * RS + KP * RA : p, *r = rows(c), *vs = vals(c) + 4 * g * WS + 16 * cw + m;
      f32x4 w, kx[KT], d[KT], pre, suf, rest;
      s16x4 ky[KT];
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = vs[e * WS];
      const f32x4 A_row = *reinterpret_cast<const f32x4*>(A + (BONUS ? row_of_token(m) : m) * RA + 4 * g);
      float total = 0.f;
      if constexpr (CHANNEL) {
        const float *kt_ = p + C * RS, *totals = A + C * RA;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
          kx[kt] = *reinterpret_cast<const f32x4*>(kt_ + (k0 + 16 * kt + m) * RA + 4 * g);
          d[kt] = *reinterpret_cast<const f32x4*>(totals + k0 + 16 * kt + 4 * g);
          if constexpr (BONUS) ky[kt] = *reinterpret_cast<const s16x4*>(reinterpret_cast<const u16*>(totals + KP) + (k0 + 16 * kt + m) * RA + 4 * g);
        }
      } else {
        const float* scalars = p + kMade - 3 * C;
        pre = *reinterpret_cast<const f32x4*>(scalars + 4 * g);
        suf = *reinterpret_cast<const f32x4*>(scalars + C + 4 * g);
        rest = *reinterpret_cast<const f32x4*>(scalars + 2 * C + 4 * g);
        total = scalars[C - 1];
        const f32x4 scale = *reinterpret_cast<const f32x4*>(r + 2 * C * RS + 4 * g);
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
          for (int e = 0; e < 4; ++e) kx[kt][e] = r[C * RS + (4 * g + e) * RS + k0 + 16 * kt + m];
        if constexpr (DELTA) {
          const float* y = ys(c) + 4 * g * WS + 16 * cw + m;
          f32x4 s;
#pragma unroll
          for (int e = 0; e < 4; ++e) s[e] = y[e * WS] + y[C * WS + e * WS];
          if constexpr (KS == 4) {
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] += y[2 * C * WS + e * WS] + y[3 * C * WS + e * WS];
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = scale[e] * (w[e] - pre[e] * s[e]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] *= scale[e];
        }
      }
      const f32x4 x = w;
      if constexpr (DELTA) w = times_rows(*reinterpret_cast<const f32x4*>(p + C * RA + m * RA + 4 * g), x);
      const bool odd = some_not_finite(w);                // (delta rule: of x, then every row of w)
      if constexpr (DELTA) {
        if (odd) w = times_rows_in_order(p + C * RA, m, g, x);
      }
      // this part's share of the results: its keys' of what the state holds, its tokens' of the chunk's own
      f32x4 first, second = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (kResults) {
        const f32x4 before = times_state((CHANNEL ? p : r) + m * RS + 4 * g);
        first = before;
        if (odd) {
          if (part == 0) second = times_rows_in_order(A, m, g, w);
          if (FORM == hxm::kChunkGated) second += before;
        } else if constexpr (BONUS) {                       // (in double: what rounding leaves over goes to the smaller number)
          f64x4 sum = f64x4{0., 0., 0., 0.};
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (e / (4 / KS) == part) sum = __builtin_amdgcn_mfma_f64_16x16x4f64((double)A_row[e], (double)w[e], sum, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            second[e] = (float)sum[e];
            first[e] += (float)(sum[e] - (double)second[e]);
          }
        } else {
          if (FORM == hxm::kChunkGated) second = before;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (e / (4 / KS) == part) second = mma4(A_row[e], w[e], second);
        }
        if constexpr (!CHANNEL) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            first[e] = before[e] * pre[e];
            second[e] += __builtin_fmaf(before[e], rest[e], __builtin_fmaf(before[e], pre[e], -first[e]));
          }
        }
      }
      if constexpr (!CHANNEL) {
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] *= suf[e];
      }
      s16x4 w16;
#pragma unroll
      for (int e = 0; e < 4; ++e) w16[e] = (short)BF16::from_float(w[e]);
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        if constexpr (BONUS) {
          const f32x4 more = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ky[kt], w16, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) st.S[kt][e] = __builtin_fmaf(st.S[kt][e], d[kt][e], more[e]);
        } else if constexpr (CHANNEL) {
          st.S[kt] *= d[kt];
        } else {
          st.S[kt] *= total;
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) st.S[kt] = mma4(kx[kt][e], w[e], st.S[kt]);
      if constexpr (!kResults) {
#pragma unroll
        for (int kt = 0; kt < (CHANNEL ? KT : 1); ++kt)
#pragma unroll
          for (int e = 0; e < 4; ++e) left[kt][e] = decayed(left[kt][e], CHANNEL ? d[kt][e] : total);
      } else {
        put(outs(c), second);
        if constexpr (FORM != hxm::kChunkGated) put(outs(c) + I::kShares, first);
      }
      if constexpr (DELTA) {
        if (c + 1 < n_chunks) put(ys(c + 1), times_state(rows(c + 1) + C * RS + m * RS + 4 * g));
      }
    }
    lds_barrier();
    if constexpr (PASS == kSegmentStates) {
      st.store(segment_at(a, (int64_t)blockIdx.z + 1, head) + (int64_t)k0 * a.V, a.K - k0, a.V, col, g);
      if (blockIdx.y == 0 && cw == 0 && m == 0) {
        double* decays = reinterpret_cast<double*>(segment_at(a, blockIdx.z, head) + segment_state(a));
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int kk = k0 + 16 * kt + 4 * g + e;
            if (kk < a.K) decays[kk] = left[CHANNEL ? kt : 0][e];
          }
      }
    } else if (last) {
      st.store(slot, a.K - k0, a.V, col, g);
    }
    return;
  }

  const int tid = (int)threadIdx.x, qk_head = head / (a.heads / a.qk_heads);
  const typename QK::storage* q = (const typename QK::storage*)a.q + t_begin * a.q_stride + (int64_t)qk_head * a.K;
  const typename QK::storage* k = (const typename QK::storage*)a.k + t_begin * a.k_stride + (int64_t)qk_head * a.K;
  const typename VT::storage* v = (const typename VT::storage*)a.v + t_begin * a.v_stride + (int64_t)head * a.V;
  const bool scaled = !BONUS && FORM != hxm::kChunkGated && (DELTA || a.vscale);
  const float* per_token = DELTA ? a.beta : a.vscale ? a.vscale : a.decay;
  const float* from = a.made + ((chunk_number(t_seq, seq) + (PASS == kWhole ? 0 : (int64_t)part_at * a.segment)) * a.heads + head) * kMade + kSkip;
  const int v_row = tid / (W / 4), v_col = tid % (W / 4) * 4;      // (16 W / 4 threads)
  const bool v_mine = 16 * W / 4 >= 256 || v_row < C;
  struct Set {
    Rows<QK, VEC, KP, 256> q, k;           // (a decay per head)
    Piece<VT, 4, VEC> v;
    MadeRows<kMade - kSkip, 256> made;
    float scale;
  } sets[kAhead];
  auto fetch = [&](Set& s, int chunk) __attribute__((always_inline)) {
    chunk = min(chunk, n_chunks - 1);
    const int n = rows_of(chunk);
    const int64_t t0 = (int64_t)chunk * C;
    if constexpr (!CHANNEL) {
      if constexpr (kResults) s.q.fetch(q + t0 * a.q_stride, a.q_stride, 0, a.K, n, tid);
      s.k.fetch(k + t0 * a.k_stride, a.k_stride, 0, a.K, n, tid);
    }
    s.made.fetch(from + (int64_t)chunk * a.heads * kMade, tid);
    s.v.load(v + (t0 + min(v_row, n - 1)) * a.v_stride, col0 + v_col, a.V);
    if constexpr (FORM == hxm::kChunkDecay || DELTA) s.scale = per_token[(t_begin + t0 + min(CHANNEL ? v_row : m, n - 1)) * a.heads + head];
  };
  auto store = [&](const Set& s, int chunk) __attribute__((always_inline)) {
    if (chunk >= n_chunks) return;
    const int n = rows_of(chunk);
    float* r = rows(chunk);
    s.made.store(made(chunk) + kSkip, tid);
    if constexpr (!CHANNEL) {
      if constexpr (kResults) s.q.store(r, 0, a.K, n, 1.f, tid);
      s.k.store(r + C * RS, 0, a.K, n, 1.f, tid);
      if (tid < C) r[2 * C * RS + row_of_token(m)] = m >= n ? (DELTA ? 0.f : 1.f) : scaled ? s.scale : 1.f;      // (a row past the portion changes nothing)
    }
    if (v_mine) {
      f32x4 f;
#pragma unroll
      for (int j = 0; j < 4; ++j) f[j] = s.v.get(j, v_row < n, col0 + v_col, a.V) * (CHANNEL && scaled ? s.scale : 1.f);
      *reinterpret_cast<f32x4*>(vals(chunk) + row_of_token(v_row) * WS + v_col) = f;
    }
  };
  // results: the parts' shares added up in double, rounded once
  auto write = [&](int chunk) __attribute__((always_inline)) {
    if constexpr (!kResults) return;
    const int col = col0 + v_col;
    if (!v_mine || v_row >= rows_of(chunk)) return;
    const float* o = outs(chunk) + row_of_token(v_row) * WS + v_col;
    f32x4 f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      double sum = o[j];
#pragma unroll
      for (int share = 1; share < I::kResult / (C * WS); ++share) sum += (double)o[share * C * WS + j];
      f[j] = (float)sum;
    }
    float* to = a.out + (t_begin + (int64_t)chunk * C + v_row) * ((int64_t)a.heads * a.V) + (int64_t)head * a.V + col;
    if (VEC) {
      if (col < a.V) *reinterpret_cast<f32x4*>(to) = f;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (col + j < a.V) to[j] = f[j];
    }
  };
#pragma unroll
  for (int i = 0; i < kAhead; ++i) fetch(sets[i], i);
  for (int c0 = -kLead; c0 < n_chunks; c0 += kAhead) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int c = c0 + i;
      if (c >= n_chunks) break;
      store(sets[i], c + kLead);
      fetch(sets[i], c + kLead + kAhead);
      if (c >= 2) write(c - 2);                           // (chunk c - 1's are being made)
      lds_barrier();
    }
  }
  if (n_chunks >= 2) write(n_chunks - 2);
  lds_barrier();
  write(n_chunks - 1);
}

// numbers that chunks may have
int64_t chunk_numbers(const ChunkScanArgs& a) { return a.n_tokens / C + a.n_seq; }
int64_t segment_numbers(const ChunkScanArgs& a, int segment) { return a.n_tokens / (C * segment) + a.n_seq; }
// With 32 value channels a workgroup every one of them has a compute unit: the keys go to four waves.  (Else twice the rows would be
// brought in for each channel: the gated form above 146 us in the chain, 115 with 64 channels.)
bool few_chains(const ChunkScanArgs& a) { return (int64_t)a.n_seq * a.heads * ((a.V + 31) / 32) <= 256; }
template <int KP>
int64_t made_floats(const ChunkScanArgs& a) {
  if (a.form == hxm::kChunkGated) return kMadeChannel<KP, hxm::kChunkGated>;
  if (a.form == hxm::kChunkBonus) return kMadeChannel<KP, hxm::kChunkBonus>;
  if (a.per_channel) return kMadeChannel<KP, hxm::kChunkDecay>;
  return a.form == hxm::kChunkDelta ? kMadeHead<true> : kMadeHead<false>;
}

template <int KP, int FORM, bool CHANNEL, int KS, typename QK, typename VT, bool VEC, int PASS>
int launch_parts(const ChunkScanArgs& a, hipStream_t s) {
  typedef Image<KP, FORM, CHANNEL, KS> I;
  const int64_t z = PASS == kWhole ? a.n_seq : segment_numbers(a, a.segment);
  return launch_chunks(chunk_chain_kernel<KP, FORM, CHANNEL, KS, QK, VT, VEC, PASS>, dim3((unsigned)a.heads, (unsigned)((a.V + I::W - 1) / I::W), (unsigned)z), 768,
                       sizeof(float) * I::kLds, a, s);
}
template <int KP, int FORM, bool CHANNEL, typename QK, typename VT, bool VEC>
int launch_chain(const ChunkScanArgs& a, hipStream_t s) {
  constexpr int KS = KP == 128 ? 4 : 2;                   // of few chains
  if constexpr (FORM != hxm::kChunkDelta) {
    if (a.segment > 0) {
      const int rc = launch_parts<KP, FORM, CHANNEL, KS, QK, VT, VEC, kSegmentStates>(a, s);
      return rc != HX_OK ? rc : launch_parts<KP, FORM, CHANNEL, KS, QK, VT, VEC, kSegmentResults>(a, s);
    }
  }
  if constexpr (KP == 128) {
    if (few_chains(a)) return launch_parts<KP, FORM, CHANNEL, KS, QK, VT, VEC, kWhole>(a, s);
  }
  if constexpr (FORM == hxm::kChunkDelta) return HX_ERR_UNSUPPORTED;      // (many chains of the delta rule take one launch: two gain nothing, chunk_scan_workspace)
  else return launch_parts<KP, FORM, CHANNEL, 2, QK, VT, VEC, kWhole>(a, s);
}
template <int KP, int FORM, typename QK, typename VT, bool VEC>
int launch_channel(const ChunkScanArgs& a, hipStream_t s) {
  const int rc = launch_chunks(chunk_channel_make_kernel<KP, FORM, QK, VEC>, dim3((unsigned)(chunk_numbers(a) * a.heads)), 256, 0, a, s);
  return rc != HX_OK ? rc : launch_chain<KP, FORM, true, F32, VT, VEC>(a, s);
}
template <int KP, int FORM, typename QK, typename VT, bool VEC>
int launch_head(const ChunkScanArgs& a, hipStream_t s) {
  constexpr bool DELTA = FORM == hxm::kChunkDelta;
  const int rc = launch_chunks(chunk_head_make_kernel<KP, DELTA, QK, VEC>, dim3((unsigned)(chunk_numbers(a) * a.heads)), 128, 0, a, s);
  return rc != HX_OK ? rc : launch_chain<KP, FORM, false, QK, VT, VEC>(a, s);
}

template <int KP, typename QK, typename VT, bool VEC>
int launch_form(const ChunkScanArgs& a, hipStream_t s) {
  if (a.form == hxm::kChunkGated) return launch_channel<KP, hxm::kChunkGated, QK, VT, VEC>(a, s);
  if (a.form == hxm::kChunkBonus) return launch_channel<KP, hxm::kChunkBonus, QK, VT, VEC>(a, s);
  if (a.per_channel) return launch_channel<KP, hxm::kChunkDecay, QK, VT, VEC>(a, s);
  if (a.form == hxm::kChunkDelta) {
    if constexpr (KP == 128) return launch_head<KP, hxm::kChunkDelta, QK, VT, VEC>(a, s);
    else return HX_ERR_UNSUPPORTED;
  }
  return launch_head<KP, hxm::kChunkDecay, QK, VT, VEC>(a, s);
}

template <typename QK, typename VT>
int launch_width(const ChunkScanArgs& a, hipStream_t s) {
  const bool vec = rows_by_four(a) && (uintptr_t)a.out % 16 == 0;
  if (a.K <= 64) return vec ? launch_form<64, QK, VT, true>(a, s) : launch_form<64, QK, VT, false>(a, s);
  return vec ? launch_form<128, QK, VT, true>(a, s) : launch_form<128, QK, VT, false>(a, s);
}

}  // namespace

namespace hxm {

static int64_t plan_made(const ChunkScanArgs& a) { return chunk_numbers(a) * a.heads * (a.K <= 64 ? made_floats<64>(a) : made_floats<128>(a)); }
static int64_t plan_floats(const ChunkScanArgs& a, int segment) {
  return plan_made(a) + (segment > 0 ? segment_numbers(a, segment) * a.heads * (segment_state(a) + 2 * a.K) : 0);
}
// Chunks a segment, 0: portions stay whole.  longest: chunks of the longest portion, or of the mean one where that is all that is known.
// Segments take a launch more and every chunk's keys twice (a chunk of the states' launch costs about 0.6 of one with results), and pay where the compute
// units have room for all of them at once: a second round costs more than longer segments (2 portions of 500 - 684 tokens, 32 heads of 128 x 128,
// gated: whole 74 us, segments of 8, 12, 16 chunks 115, 110, 103).  So a segment is as short as that room allows, at least 6 chunks (96 tokens; at 4
// the launches around them cost as much) and a seventh of the portion, as the last segment's start is put together out of all before it (8 heads of 128 x 128, 1151
// tokens in segments of 4, 8, 12, 16 chunks 81, 53, 47, 50 us, whole 83).
// Whole and in segments, us: gated, 3 of 54 - 839 tokens, 8 heads of 64 x 64 57 36; bonus form, one of 1002, 16 heads of 64 x 64 87 44; decayed
// sum, one of 1100, 8 of 128 x 128 84 40.  In 110 batches of 1 to 10 portions 0.89 of the time in the mean (the best
// length of each would be 0.87), none slower.  Errors against 64 bits are the same to the third digit (a chain rounds as often as its segments do).
static int segment_chunks(const ChunkScanArgs& a, double longest) {
  if (a.form == kChunkDelta) return 0;                    // (what a chunk leaves of a state is a matrix there)
  const int64_t columns = a.heads * (int64_t)((a.V + (a.K <= 64 ? 63 : 31)) / (a.K <= 64 ? 64 : 32)), room = 256 / columns - a.n_seq;
  if (room < 1) return 0;
  const int64_t fits = a.n_tokens / (C * (room + 1)) + 1;      // the least with n_tokens / (16 segment) <= room
  const int64_t segment = std::max<int64_t>({6, fits, (int64_t)std::ceil(longest / 7)});
  return longest >= 1.6 * segment + 6 ? (int)segment : 0;
}
// Whether a call takes the launches of this file: the chunks of a segment (0: whole portions), -1: it does not
static int chain_plan(const ChunkScanArgs& a) {
  if (!chunk_scan_fits(a) || (a.V + 31) / 32 > 65535 || (a.form == kChunkDelta && a.K <= 64)) return -1;
  if (chunk_numbers(a) * a.heads > INT32_MAX || plan_floats(a, 0) > (int64_t)1 << 28) return -1;      // (1 GiB)
  // Two launches save `few` or `many` us for a chunk of the chain and take `cost` us for each chunk and head, and 2 us.  Fitted to 12 batches
  // of 1 to 16 portions of 64 to 1151 tokens, 8 to 32 heads and 12 forms and sizes; one launch and two, us, about the line: delta rule, 128 x 128, 32
  // heads: 2 portions of 128 27 28, 2 of 600 104 91, 16 heads: 4 of 1000 167 143; decayed sum, 128 x 64, 32 heads: 4 of 256 40 33, 8 of 512 74 79;
  // 64 x 64: one of 1151 92 86, 4 of 1000 83 86; gated form, 128 x 128, 32 heads: 4 of 64 21 23, 4 of 256 57 53; 64 x 64: 4 of 1000 115 97, 8 of 512 71
  // 83; bonus form, 128 x 128, 16 heads: 4 of 1000 162 121, 8 of 512 95 98; 64 x 64, 8 heads: 8 of 512 52 55; a decay per channel, 128 x 64, 32 heads: 4 of 256 45
  // 39, 8 of 512 89 123.
  // (One decay a head: fitted against one launch of sixteen tokens at a time, which float q and k of a decayed sum still take.  Against chunk_head.hip, thirty-two
  // at a time, two launches are as fast or faster up to 128 workgroups — one of 1100, 16 heads of 128 x 128: delta rule 138 and 157, decayed sum of bfloat16 q
  // and k 87 and 98 — and up to 7 % behind at 256: 4 of 1000, 32 heads of 128 x 64: 177 and 165, 108 and 101.  Not fitted anew for those; the decayed sum's
  // results are less off in two, 0.78 and 0.86 e-7.)
  // (And one launch takes 20 us: shorter calls are bound by their caller, who would have to ask for a workspace: 19.2 and 21.7 us.)
  struct Line { double few, many, cost, one; };           // few: keys dealt to four waves; one: us a chunk in one launch
  const bool wide = a.K > 64;
  const Line line = a.form == kChunkGated   ? (wide ? Line{1.5, 1.05, 0.0067, 2.6} : Line{0.6, 0.6, 0.003, 1.6})
                    : a.form == kChunkBonus ? (wide ? Line{1.1, 0.6, 0.008, 2.4} : Line{0.15, 0.15, 0.0027, 1.5})
                    : a.form == kChunkDelta ? Line{0.65, 0.0, 0.0044, 2.7}
                    : a.per_channel         ? (wide ? Line{1.15, 1.0, 0.0085, 2.3} : Line{0.2, 0.2, 0.003, 1.4})
                                            : (wide ? Line{0.78, 0.3, 0.0025, 2.0} : Line{0.1, 0.1, 0.0009, 1.3});
  const double mean = (double)a.n_tokens / a.n_seq / C, longest = a.longest > 0 ? (double)a.longest / C : mean;
  const int64_t chains = (int64_t)a.n_seq * a.heads * ((a.V + VW - 1) / VW);      // a compute unit takes one at a time
  const double chain = chains <= 256 ? longest : mean * ((chains + 255) / 256), saved = (few_chains(a) ? line.few : line.many) * chain;
  const bool whole = chain * line.one >= 20.0 && saved > line.cost * a.n_tokens / C * a.heads + 3.5;
  // (Decayed sums of bfloat16 q and k with one decay a head that one launch of chunk_head.hip would serve stay there: segments of sixteen tokens at a time are up to twice as fast, but leave
  // states off by up to a tenth more where the last chunk is short: one portion of 483, 8 heads of 64 x 64, 37 and 28 us, 6.1 and 6.7e-8.)
  const bool by_parts = a.form == kChunkDecay && !a.per_channel && a.q_dtype == HX_BF16 && a.k_dtype == HX_BF16;
  const int segment = by_parts && !whole ? 0 : segment_chunks(a, longest);
  if (segment > 0 && plan_floats(a, segment) <= (int64_t)1 << 28) return segment;
  return whole ? 0 : -1;
}

int64_t chunk_scan_workspace(const ChunkScanArgs& a) {
  const int segment = chain_plan(a);
  return segment < 0 ? 0 : plan_floats(a, segment);
}

int chunk_chain(const ChunkScanArgs& args, hipStream_t s) {
  ChunkScanArgs a = args;
  const int segment = chain_plan(a);
  a.segment = segment > 0 ? segment : 0;
  a.segments = a.made + plan_made(a);
  if (a.q_dtype == HX_BF16) return launch_width<BF16, BF16>(a, s);
  return a.v_dtype == HX_F32 ? launch_width<F32, F32>(a, s) : launch_width<F32, BF16>(a, s);
}

}  // namespace hxm
