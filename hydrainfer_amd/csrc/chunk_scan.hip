// chunk_scan.hip — a recurrence with a matrix state S [K, V] per head and sequence over portions of prompts, sixteen tokens at a
// time, all of it in float (v_mfma_f32_16x16x4_f32, an ascending chain of fused multiply-adds) or wider.  With S the state before the
// chunk and products of decays only — never a quotient, so that decays that vanish give zeros and not 0 / 0:
//     Y = (K * prefix) S                            delta rule: what the chunk's keys read from the old state
//     W = M (b (V - Y)), M = (I + b (K K^T) L)^-1   delta rule (strictly lower part; M by substitution); else W = s V
//     O = (Q * prefix) S + A W                      A[t, s] = sum_d q_t[d] k_s[d] prod(s < r <= t) a_r[d] for s <= t
//     S <- total S + (K * suffix)^T W               prefix / suffix / total: products of the decays up to t / behind s / of the chunk
// Token by token the scan is bound by the vector ALU (three operations a state element and token); here the state's elements
// pass through the matrix cores at four times that rate, and what is left to the vector ALU does not depend on V.
//
// A workgroup owns 64 value channels of one (sequence, head): four consumer waves hold the state, 16 channels of values and all
// of the keys each, as accumulators (rows 4 (lane / 16) + e, column lane % 16) — which is at the same time the operand of the
// products with S when the sum over key channels is taken in the order 16 tile + 4 (lane / 16) + e, so the state never leaves
// its registers.  Producer waves work one chunk ahead (A, M, prefixes, suffixes) and bring rows in two chunks ahead, requested
// three chunks before that from clamped addresses; one workgroup barrier a chunk.  The workgroups of a sequence stand next to
// each other: a long portion among short ones is spread over all XCDs (dealt round robin).
//   per head:    chunk_head_kernel — Q K^T and K K^T on the matrix cores, decays as factors of the accumulators' rows.  (Thirty-two tokens at
//                a time, in bfloat16 parts, where that is faster: chunk_head.hip.)
//   per channel: chunk_channel_kernel — A by running products over the tokens on the vector ALU, a lane one or two key channels,
//                summed over the wave by a transposing butterfly that leaves one element of A in every second lane.
// What bounds it now: the chunks of a sequence follow each other (2.5 us each with states of 128 x 128; 1.8 us of float matrix
// products on the SIMDs that hold a consumer and a maker of A or M).  Measured against one token at a time, 4 portions of 797 -
// 1151 tokens: delta rule, 32 heads of 128 x 128, 479 -> 189 us; bonus form, 32 heads of 64 x 64, 207 -> 105 us; gated form, 32 heads of 128 x 128, 720 -> 205 us with its norm (171 in the two launches of chunk_chain.hip, which
// batches of few chains for their length take).
// What the rounding costs: a token at a time rounds a state's element once a token, and each rounding decays with the state.  Here
// the products of decays, of keys with them and the chunk's sums are rounded besides, and four things keep that from showing: sums
// over tokens run from the first token to the last and on top of the decayed state (row_of_token); products of decays carry what
// their roundings leave over (Product); sums over key channels are cut in eight or sixteen chains; and the bonus form, whose
// k v is often exact, adds up within a chunk in double and keeps the rest of its suffixed keys.  Error against 64 bits (2-norm), a
// token at a time and here, 3 portions of 200 - 600 tokens, 16 heads of 128 x 128 (64 x 64): results delta 1.07 1.07 (1.00 1.00),
// decay 1.04 0.84 (0.97 0.77), bonus 0.90 0.82 (0.83 0.77) e-7; states delta 0.74 0.73 (0.75 0.74), decay 0.68 0.62 (0.72
// 0.66), bonus 0.46 0.45 (0.47 0.45), gated 1.42 1.09 (1.41 1.08) e-7.
#include <cmath>

#include "chunk_parts.h"

namespace {

// (for the scheduler) FIRST reads from LDS, then a read behind every PER products, N times, then REST products: left alone it
// asks for two rows and waits for them after every eight products.  Tuned by measuring, 4 portions of 797 - 1151 tokens and 32 heads:
// delta rule 128 x 128 207 us without, 189 here (<6, 28, 2, 12> 200, <12, 22, 3, 3> 214), 64 x 64 126 and 122; bonus form 64 x 64
// 115 and 105.  The gated form, bound by its producers, gains nothing.
template <int FIRST, int N, int PER, int REST>
__device__ __forceinline__ void products_behind_reads() {
  __builtin_amdgcn_sched_group_barrier(0x100, FIRST, 0);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, PER, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
  }
  __builtin_amdgcn_sched_group_barrier(0x008, REST, 0);
}

// ---------------------------------------------------------------------------------------------------------------
// One decay per token and head.
// ---------------------------------------------------------------------------------------------------------------
template <int KP, bool DELTA, typename QK, typename VT, bool VEC>
__global__ __launch_bounds__(512) void chunk_head_kernel(ChunkScanArgs a) {
  constexpr int KT = KP / 16, RS = KP + 4;
  constexpr int kRaw = 2 * C * RS + C * VS + 3 * C;       // q | k | v | decay, value scale, write strength
  constexpr int kMade = 2 * C * RA + 3 * C;               // A | M (T while it is made) | prefix, suffix, what the prefix's rounding left over
  extern __shared__ __attribute__((aligned(16))) float lds[];      // raw[3] | made[2]
  const int seq = blockIdx.z, head = blockIdx.x, col0 = (int)blockIdx.y * VW;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, m = lane & 15;
  const int64_t t_begin = a.q_cu[seq];
  const int n_tok = (int)(a.q_cu[seq + 1] - t_begin);
  if (n_tok <= 0) return;                                 // (the whole workgroup)
  const int n_chunks = (n_tok + C - 1) / C;
  float* slot = a.state + (int64_t)a.slots[seq] * a.slot_stride + (int64_t)head * a.K * a.V;
  auto raw = [&](int chunk) { return lds + chunk % 3 * kRaw; };
  auto made = [&](int chunk) { return lds + 3 * kRaw + (chunk & 1) * kMade; };
  auto rows_of = [&](int chunk) { return min(C, n_tok - chunk * C); };

  if (wave >= 4) {
    const int cw = wave - 4, col = col0 + 16 * cw + m;
    State<KT> st;
    st.load(slot, a.K, a.V, col, g, a.positions[t_begin] == 0);
    lds_barrier();
    lds_barrier();
    for (int c = 0; c < n_chunks; ++c) {
      const float* r = raw(c);
      const float *q = r + m * RS + 4 * g, *k = r + C * RS + m * RS + 4 * g, *vs = r + 2 * C * RS, *sc = vs + C * VS;
      const float* A = made(c);
      const float* M = A + C * RA;
      const f32x4 pre = *reinterpret_cast<const f32x4*>(M + C * RA + 4 * g), suf = *reinterpret_cast<const f32x4*>(M + C * RA + C + 4 * g);
      const f32x4 rest = *reinterpret_cast<const f32x4*>(M + C * RA + 2 * C + 4 * g);
      const float total = M[C * RA + C - 1];
      f32x4 x, w;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = vs[(4 * g + e) * VS + 16 * cw + m];
      if constexpr (DELTA) {
        const f32x4 y = st.times(k), b = *reinterpret_cast<const f32x4*>(sc + 2 * C + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = b[e] * (x[e] - pre[e] * y[e]);
        w = times_rows(*reinterpret_cast<const f32x4*>(M + m * RA + 4 * g), x);
      } else {
        const f32x4 s = *reinterpret_cast<const f32x4*>(sc + C + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = x[e] * s[e];
      }
      const f32x4 before = st.times(q);
      f32x4 within = times_rows(*reinterpret_cast<const f32x4*>(A + m * RA + 4 * g), w);
      if constexpr (KP == 128) products_behind_reads<8, 26, 3, 1>();
      else products_behind_reads<10, 9, 3, 13>();
      if (some_not_finite(w)) {                            // (of x: then every row of w)
        if constexpr (DELTA) w = times_rows_in_order(M, m, g, x);
        within = times_rows_in_order(A, m, g, w);
      }
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = __builtin_fmaf(before[e], pre[e], __builtin_fmaf(before[e], rest[e], within[e]));
      const int n = rows_of(c);
      const int64_t t0 = t_begin + (int64_t)c * C;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (4 * e + g < n && col < a.V) a.out[(t0 + 4 * e + g) * ((int64_t)a.heads * a.V) + (int64_t)head * a.V + col] = o[e];
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] *= suf[e];
      const float* kr = r + C * RS + 4 * g * RS + m;      // k of row 4 g + e, channel 16 kt + m
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        st.S[kt] *= total;
#pragma unroll
        for (int e = 0; e < 4; ++e) st.S[kt] = mma4(kr[e * RS + 16 * kt], w[e], st.S[kt]);
      }
      products_behind_reads<16, 16, 2, 1>();
      lds_barrier();
    }
    st.store(slot, a.K, a.V, col, g);
    return;
  }

  // Producers: wave 0 A, prefixes and suffixes, wave 1 M, wave 2 brings q and the values, wave 3 k and the tokens' scalars.
  const int qk_head = head / (a.heads / a.qk_heads);
  // (x k^T)[i, j] with rows i = 4 g + e and column j = m: tokens 4 e + g and t_m; N chains
  const int t_m = row_of_token(m);
  auto with_keys = [&](const float* rows_x, const float* k, auto chains) __attribute__((always_inline)) {
    constexpr int N = decltype(chains)::value;
    f32x4 p[N];
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
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
  };
  auto decays = [&](const float* sc, float (&d)[C]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < C / 4; ++i) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(sc + 4 * i);
#pragma unroll
      for (int e = 0; e < 4; ++e) d[4 * i + e] = x[e];
    }
  };
  // A, prefixes and suffixes: with sixteen chains and products of decays rounded once, as A's rounding is the larger part of a
  // result's error
  auto finish_A = [&](int chunk) __attribute__((always_inline)) {
    const float* r = raw(chunk);
    float* A = made(chunk);
    const f32x4 xk = with_keys(r, r + C * RS, std::integral_constant<int, 16>());
    float d[C];
    decays(r + 2 * C * RS + C * VS, d);
    Product run, mine[4];                                 // run = prod(t_m < r <= t) d_r, kept at the lane's four rows
#pragma unroll
    for (int t = 0; t < C; ++t) {
      run.by(t > t_m ? d[t] : 1.f);
      const bool here = (t & 3) == 0 || (t & 3) == g;
      mine[t >> 2].hi = here ? run.hi : mine[t >> 2].hi;
      mine[t >> 2].lo = here ? run.lo : mine[t >> 2].lo;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) A[(4 * g + e) * RA + m] = t_m <= 4 * e + g ? mine[e].times(xk[e]) : 0.f;
    if (g == 0) A[2 * C * RA + C + m] = run.value();      // behind token t_m
    if (m == 0) {                                         // up to the rows' tokens: the first one's decay and all behind it
      f32x4 prefix, rest;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        prefix[e] = mine[e].times(d[0]);
        rest[e] = mine[e].rest(d[0], prefix[e]);
      }
      *reinterpret_cast<f32x4*>(A + 2 * C * RA + 4 * g) = prefix;
      *reinterpret_cast<f32x4*>(A + 2 * C * RA + 2 * C + 4 * g) = rest;
    }
  };
  auto finish_M = [&](int chunk) __attribute__((always_inline)) {
    const float *k = raw(chunk) + C * RS, *sc = k + C * RS + C * VS;
    float* A = made(chunk) + C * RA;                      // T (by tokens), then M
    const f32x4 xk = with_keys(k, k, std::integral_constant<int, 4>());
    float d[C], run = 1.f, mine[4];
    decays(sc, d);
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
  };
  if (wave < 2) {
    for (int c = -2; c < n_chunks; ++c) {
      if (c + 1 >= 0 && c + 1 < n_chunks) {
        if (wave == 0) finish_A(c + 1);
        else if constexpr (DELTA) finish_M(c + 1);
      }
      lds_barrier();
    }
    return;
  }
  // Rows come in kAhead chunks ahead of the interval that puts them in LDS: an interval is shorter than a load's way.  Behind
  // the last chunk the last one comes again.
  const typename QK::storage* x = (const typename QK::storage*)(wave == 2 ? a.q : a.k) + t_begin * (wave == 2 ? a.q_stride : a.k_stride) + (int64_t)qk_head * a.K;
  const int64_t x_stride = wave == 2 ? a.q_stride : a.k_stride;
  const typename VT::storage* v = (const typename VT::storage*)a.v + t_begin * a.v_stride + (int64_t)head * a.V;
  const float* per_token[3] = {a.decay, a.vscale ? a.vscale : a.decay, DELTA ? a.beta : a.decay};
  struct Set {
    Rows<QK, VEC, KP, 64> rows;
    Rows<VT, VEC, VW, 128> values;         // (waves 2 and 3 half of them each)
    float scalars[3];
  } sets[kAhead];
  auto fetch = [&](Set& s, int chunk) __attribute__((always_inline)) {
    chunk = min(chunk, n_chunks - 1);
    const int n = rows_of(chunk);
    s.rows.fetch(x + (int64_t)chunk * C * x_stride, x_stride, 0, a.K, n, lane);
    s.values.fetch(v + (int64_t)chunk * C * a.v_stride, a.v_stride, col0, a.V, n, (int)threadIdx.x - 128);
    const int64_t th = (t_begin + chunk * C + min(m, n - 1)) * a.heads + head;
#pragma unroll
    for (int i = 0; i < 3; ++i) s.scalars[i] = per_token[i][th];
  };
  auto store = [&](const Set& s, int chunk) __attribute__((always_inline)) {
    if (chunk >= n_chunks) return;
    const int n = rows_of(chunk);
    float* r = raw(chunk);
    s.rows.store(r + (wave == 2 ? 0 : C * RS), 0, a.K, n, 1.f, lane);
    s.values.store(r + 2 * C * RS, col0, a.V, n, 1.f, (int)threadIdx.x - 128);
    if (wave == 3 && g == 0) {             // (a row past the portion changes nothing)
      float* sc = r + 2 * C * RS + C * VS;                 // (decays by token, the others by row)
      sc[m] = m < n ? s.scalars[0] : 1.f;
      sc[C + row_of_token(m)] = m < n && a.vscale ? s.scalars[1] : 1.f;
      sc[2 * C + row_of_token(m)] = m < n && DELTA ? s.scalars[2] : 0.f;
    }
  };
#pragma unroll
  for (int i = 0; i < kAhead; ++i) fetch(sets[i], i);
  for (int c0 = -2; c0 < n_chunks; c0 += kAhead) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int c = c0 + i;
      if (c >= n_chunks) break;
      store(sets[i], c + 2);
      fetch(sets[i], c + 2 + kAhead);
      lds_barrier();
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// One decay per token and key channel.
// ---------------------------------------------------------------------------------------------------------------
template <int KP, int FORM, typename QK, typename VT, bool VEC>
__global__ __launch_bounds__(768) void chunk_channel_kernel(ChunkScanArgs a) {
  constexpr int KT = KP / 16, RS = KP + 4, NP = KP / 64;  // NP key channels a lane of a producer wave
  constexpr bool GATED = FORM == hxm::kChunkGated, BONUS = FORM == hxm::kChunkBonus;
  constexpr int kGate = kGateFloats<KP, FORM>, kMade = kMadeChannel<KP, FORM>;
  extern __shared__ __attribute__((aligned(16))) float lds[];      // gates[2] | made[2] | values[3]
  const int seq = blockIdx.z, head = blockIdx.x, col0 = (int)blockIdx.y * VW;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, m = lane & 15;
  const int64_t t_begin = a.q_cu[seq];
  const int n_tok = (int)(a.q_cu[seq + 1] - t_begin);
  if (n_tok <= 0) return;                                 // (the whole workgroup)
  const int n_chunks = (n_tok + C - 1) / C;
  float* slot = a.state + (int64_t)a.slots[seq] * a.slot_stride + (int64_t)head * a.K * a.V;
  auto gates = [&](int chunk) { return lds + (chunk & 1) * kGate; };
  auto made = [&](int chunk) { return lds + 2 * kGate + (chunk & 1) * kMade; };
  auto vals = [&](int chunk) { return lds + 2 * kGate + 2 * kMade + chunk % 3 * (C * VS); };
  auto rows_of = [&](int chunk) { return min(C, n_tok - chunk * C); };

  if (wave >= 4 && wave < 8) {
    const int cw = wave - 4, col = col0 + 16 * cw + m;
    State<KT> st;
    st.load(slot, a.K, a.V, col, g, a.positions[t_begin] == 0);
    lds_barrier();
    lds_barrier();
    for (int c = 0; c < n_chunks; ++c) {
      const float* p = made(c);
      const float *kt_ = p + C * RS, *A = kt_ + KP * RA, *total = A + C * RA;
      const float* vs = vals(c) + 4 * g * VS + 16 * cw + m;
      f32x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = vs[e * VS];
      const f32x4 before = st.times(p + m * RS + 4 * g);
      s16x4 w16;
#pragma unroll
      for (int e = 0; e < 4; ++e) w16[e] = (short)BF16::from_float(w[e]);
      f32x4 o = BONUS ? times_rows_double(*reinterpret_cast<const f32x4*>(A + row_of_token(m) * RA + 4 * g), w, before) : times_rows(*reinterpret_cast<const f32x4*>(A + m * RA + 4 * g), w, before);
      if constexpr (!GATED) products_behind_reads<10, 4, 4, 20>();
      if (some_not_finite(w)) o = before + times_rows_in_order(A, m, g, w);
      const int n = rows_of(c);
      const int64_t t0 = t_begin + (int64_t)c * C;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (4 * e + g < n && col < a.V) a.out[(t0 + 4 * e + g) * ((int64_t)a.heads * a.V) + (int64_t)head * a.V + col] = o[e];
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        const f32x4 d = *reinterpret_cast<const f32x4*>(total + 16 * kt + 4 * g);
        const f32x4 x = *reinterpret_cast<const f32x4*>(kt_ + (16 * kt + m) * RA + 4 * g);
        if constexpr (BONUS) {
          const s16x4 y = *reinterpret_cast<const s16x4*>(reinterpret_cast<const u16*>(total + KP) + (16 * kt + m) * RA + 4 * g);
          const f32x4 rest = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(y, w16, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) st.S[kt][e] = __builtin_fmaf(st.S[kt][e], d[e], rest[e]);
        } else {
          st.S[kt] *= d;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) st.S[kt] = mma4(x[e], w[e], st.S[kt]);
      }
      if constexpr (!GATED) products_behind_reads<6, 10, 2, 12>();
      lds_barrier();
    }
    st.store(slot, a.K, a.V, col, g);
    return;
  }

  const typename VT::storage* vp = (const typename VT::storage*)a.v + t_begin * a.v_stride + (int64_t)head * a.V;
  const float* sp = FORM == hxm::kChunkDecay ? (a.vscale ? a.vscale : a.decay) + t_begin * a.heads + head : nullptr;
  typedef Rows<VT, VEC, VW, 256> Values;
  auto fetch_values = [&](Values& x, float& scale, int chunk, int n, int tid) __attribute__((always_inline)) {
    const int64_t t0 = (int64_t)chunk * C;
    x.fetch(vp + t0 * a.v_stride, a.v_stride, col0, a.V, n, tid);
    if constexpr (FORM == hxm::kChunkDecay) scale = sp[(t0 + min(x.row_of(0, tid), n - 1)) * a.heads];
  };
  auto store_values = [&](const Values& x, float scale, int chunk, int n, int tid) __attribute__((always_inline)) {
    x.store(vals(chunk), col0, a.V, n, FORM == hxm::kChunkDecay && a.vscale ? scale : 1.f, tid);
  };
  // Producers, four waves that bring rows in and four that finish them: wave w (modulo 4) owns tokens 4 w .. 4 w + 3 of a chunk
  // (and their columns of A), lane l key channels NP l ..
  const int qk_head = GATED ? head : head / (a.heads / a.qk_heads);
  const int d0 = NP * lane;
  const ChannelBias<NP, FORM> own(a, head, d0);
  if (wave >= 8) {
    const int tid = (int)threadIdx.x - 512;
    struct Set {
      GateRows<KP, FORM, QK, VEC> rows;
      Values values;
      float s;
    } sets[kAhead];
    const typename QK::storage* qp = (const typename QK::storage*)a.q + t_begin * a.q_stride + (int64_t)qk_head * a.K;
    const typename QK::storage* kp = (const typename QK::storage*)a.k + t_begin * a.k_stride + (int64_t)qk_head * a.K;
    const int64_t d_stride = (int64_t)a.heads * a.K;
    const float* dp = GATED ? nullptr : a.decay + t_begin * d_stride + (int64_t)head * a.K;
    // (straight requests, kAhead chunks ahead; behind the last chunk the last one comes again)
    auto fetch = [&](Set& x, int chunk) __attribute__((always_inline)) {
      chunk = min(chunk, n_chunks - 1);
      const int64_t t0 = (int64_t)chunk * C;
      x.rows.fetch(qp + t0 * a.q_stride, a.q_stride, kp + t0 * a.k_stride, a.k_stride, GATED ? nullptr : dp + t0 * d_stride, d_stride, rows_of(chunk), a.K, wave - 8, d0);
      fetch_values(x.values, x.s, chunk, rows_of(chunk), tid);
    };
    auto store = [&](const Set& x, int chunk) __attribute__((always_inline)) {
      if (chunk >= n_chunks) return;
      x.rows.store(gates(chunk), own, rows_of(chunk), a.K, wave - 8, d0);
      store_values(x.values, x.s, chunk, rows_of(chunk), tid);
    };
#pragma unroll
    for (int i = 0; i < kAhead; ++i) fetch(sets[i], i);
    for (int c0 = -2; c0 < n_chunks; c0 += kAhead) {
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {
        const int c = c0 + i;
        if (c >= n_chunks) break;
        store(sets[i], c + 2);
        fetch(sets[i], c + 2 + kAhead);
        lds_barrier();
      }
    }
    return;
  }
  // the parts of A above its diagonal are never written again
  for (int i = threadIdx.x; i < C * RA; i += 256) {
    made(0)[C * RS + KP * RA + i] = 0.f;
    made(1)[C * RS + KP * RA + i] = 0.f;
  }
  const int to = place_in_A(wave, lane);
  for (int c = -2; c < n_chunks; ++c) {
    if (c + 1 >= 0 && c + 1 < n_chunks) finish_chunk<KP, FORM>(gates(c + 1), made(c + 1), own, to, wave, lane);
    lds_barrier();
  }
}

template <typename Kernel>
int launch(Kernel kernel, int threads, size_t lds, const ChunkScanArgs& a, hipStream_t s) {
  return launch_chunks(kernel, dim3((unsigned)a.heads, (unsigned)((a.V + VW - 1) / VW), (unsigned)a.n_seq), threads, lds, a, s);
}

template <int KP, int FORM, typename QK, typename VT, bool VEC>
int launch_channel(const ChunkScanArgs& a, hipStream_t s) {
  const size_t lds = sizeof(float) * (2 * kGateFloats<KP, FORM> + 2 * kMadeChannel<KP, FORM> + 3 * C * VS);
  return launch(chunk_channel_kernel<KP, FORM, QK, VT, VEC>, 768, lds, a, s);
}

template <int KP, typename QK, typename VT, bool VEC>
int launch_form(const ChunkScanArgs& a, hipStream_t s) {
  if (a.form == hxm::kChunkGated) return launch_channel<KP, hxm::kChunkGated, QK, VT, VEC>(a, s);
  if (a.form == hxm::kChunkBonus) return launch_channel<KP, hxm::kChunkBonus, QK, VT, VEC>(a, s);
  if (a.per_channel) return launch_channel<KP, hxm::kChunkDecay, QK, VT, VEC>(a, s);
  const size_t lds = sizeof(float) * (3 * (2 * C * (KP + 4) + C * VS + 3 * C) + 2 * (2 * C * RA + 3 * C));
  if (a.form == hxm::kChunkDelta) return launch(chunk_head_kernel<KP, true, QK, VT, VEC>, 512, lds, a, s);
  return launch(chunk_head_kernel<KP, false, QK, VT, VEC>, 512, lds, a, s);
}

template <typename QK, typename VT>
int launch_width(const ChunkScanArgs& a, hipStream_t s) {
  const bool vec = rows_by_four(a);
  if (a.K <= 64) return vec ? launch_form<64, QK, VT, true>(a, s) : launch_form<64, QK, VT, false>(a, s);
  return vec ? launch_form<128, QK, VT, true>(a, s) : launch_form<128, QK, VT, false>(a, s);
}

}  // namespace

namespace hxm {

bool chunk_scan_fits(const ChunkScanArgs& a) {
  // the delta rule with a decay per channel and the bonus form with one per head have no chunk form; q and k of one type, and
  // bfloat16 q and k come with bfloat16 v
  const bool types = a.q_dtype == a.k_dtype && (a.q_dtype == HX_F32 || a.v_dtype == HX_BF16);
  return types && a.K <= 128 && a.n_seq <= 65535 && (a.V + VW - 1) / VW <= 65535 && !(a.form == kChunkDelta && a.per_channel) &&
         !(a.form == kChunkBonus && !a.per_channel);
}

// One decay a head: thirty-two tokens at a time (chunk_head.hip)?  Of the time here:
//   delta rule, up to 64 key channels: no (16 portions of 60 tokens, 32 heads of 64 x 64 22.1 us here and 24.1, 4 of 797 - 1151 124 and 122, 12 of 300 - 900 124
//     and 130; there two workgroups do not share a compute unit);
//   decayed sum of float q and k, which are split in three parts: no (up to 64 key channels 1.05 - 1.5 in all of 150 batches; more, 0.95 in long portions, 1.1 -
//     1.28 in short ones);
//   bfloat16 q and k, one part each, more than 64 key channels: yes (0.67 - 1.03);
//   the rest where the tokens that a portion has in the mean fill chunks of thirty-two well enough, which take 1.7 of one of sixteen (delta rule, float: 6 - 16
//     tokens 1.17, 17 - 32 0.94, 33 - 48 1.07, 49 - 64 0.9, long ones 0.87 - 0.94) or 1.85 (decayed sum, bfloat16, up to 64 channels: up to 1.06, 0.9, 1, 0.97, 0.92).
// Rows of a chunk are addressed by 32-bit offsets there: strides of 2^28 elements and more come here.
bool by_thirty_two(const ChunkScanArgs& a) {
  const bool wide = a.K > 64, delta = a.form == kChunkDelta, parts = a.q_dtype == HX_F32;
  const bool near_rows = a.q_stride < (1 << 28) && a.k_stride < (1 << 28) && a.v_stride < (1 << 28);
  if (a.per_channel || a.form == kChunkGated || !(delta ? wide : !parts) || !near_rows) return false;
  const double mean = (double)a.n_tokens / a.n_seq;
  return (wide && !parts) || (parts ? 1.7 : 1.85) * ceil(mean / (2 * C)) < ceil(mean / C);
}

int chunk_scan(const ChunkScanArgs& a, hipStream_t s) {
  if (a.made) return chunk_chain(a, s);
  if (by_thirty_two(a)) return chunk_head(a, s);
  if (a.q_dtype == HX_BF16) return launch_width<BF16, BF16>(a, s);
  return a.v_dtype == HX_F32 ? launch_width<F32, F32>(a, s) : launch_width<F32, BF16>(a, s);
}

}  // namespace hxm
