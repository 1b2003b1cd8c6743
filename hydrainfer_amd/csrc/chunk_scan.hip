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
//   per head:    chunk_head_kernel — Q K^T and K K^T on the matrix cores, decays as factors of the accumulators' rows.
//   per channel: chunk_channel_kernel — A by running products over the tokens on the vector ALU, a lane one or two key channels,
//                summed over the wave by a transposing butterfly that leaves one element of A in every second lane.
// What bounds it now: the chunks of a sequence follow each other (2.5 us each with states of 128 x 128; 1.8 us of float matrix
// products on the SIMDs that hold a consumer and a maker of A or M).  Measured against one token at a time, 4 portions of 797 -
// 1151 tokens: delta rule, 32 heads of 128 x 128, 479 -> 189 us; decayed sum, 64 heads of 128 x 64, 432 -> 143 us; bonus form, 32
// heads of 64 x 64, 207 -> 105 us; gated form, 32 heads of 128 x 128, 720 -> 205 us with its norm.
// What the rounding costs: a token at a time rounds a state's element once a token, and each rounding decays with the state.  Here
// the products of decays, of keys with them and the chunk's sums are rounded besides, and four things keep that from showing: sums
// over tokens run from the first token to the last and on top of the decayed state (row_of_token); products of decays carry what
// their roundings leave over (Product); sums over key channels are cut in eight or sixteen chains; and the bonus form, whose
// k v is often exact, adds up within a chunk in double and keeps the rest of its suffixed keys.  Error against 64 bits (2-norm), a
// token at a time and here, 3 portions of 200 - 600 tokens, 16 heads of 128 x 128 (64 x 64): results delta 1.07 1.07 (1.00 1.00),
// decay 1.04 0.84 (0.97 0.77), bonus 0.90 0.82 (0.83 0.77) e-7; states delta 0.74 0.73 (0.75 0.74), decay 0.68 0.62 (0.72
// 0.66), bonus 0.46 0.45 (0.47 0.45), gated 1.42 1.09 (1.41 1.08) e-7.
#include <type_traits>
#include "chunk_scan.h"
#include "mix_rows.h"

namespace hxm {
int& last_hip_error();
int check_launch();
}  // namespace hxm

namespace {

using namespace hx;
using hxm::ChunkScanArgs;

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
constexpr int C = 16;             // tokens a chunk
constexpr int RA = C + 4;         // floats per row of a token by token matrix in LDS
constexpr int VW = 64;            // value channels a workgroup
constexpr int VS = VW + 4;        // floats per row of a chunk's values in LDS
constexpr int kAhead = 3;         // chunks whose rows are on their way

// Where token t of a chunk stands in LDS and in the accumulators: an instruction that sums over tokens takes rows e, 4 + e, 8 + e and
// 12 + e, one a lane group, in this order, and they are tokens 4 e .. 4 e + 3 this way.  Sums over tokens thus grow from the first
// to the last, as they do a token at a time: what has decayed is small when it is rounded.  (Its own inverse.)
__device__ __forceinline__ constexpr int row_of_token(int t) { return (t & 3) << 2 | t >> 2; }

__device__ __forceinline__ f32x4 mma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// N channels c .. of a row of n_ch on their way from global memory, as they came and from clamped addresses: no branch stands
// between two requests (the wait for one would then be a wait for all of them), and what lies past the row is masked where
// it is used.  VEC: one load (n_ch, the stride and the pointer allow it).
template <typename A, int N, bool VEC>
struct Piece {
  typedef typename A::storage T;
  typedef T vec_t __attribute__((ext_vector_type(N < 2 ? 2 : N)));
  T r[N];
  __device__ __forceinline__ void load(const T* row, int c, int n_ch) {
    if constexpr (VEC && N > 1) {
      const vec_t v = *reinterpret_cast<const vec_t*>(row + (c < n_ch ? c : 0));
#pragma unroll
      for (int j = 0; j < N; ++j) r[j] = v[j];
    } else {
#pragma unroll
      for (int j = 0; j < N; ++j) r[j] = row[c + j < n_ch ? c + j : 0];
    }
  }
  __device__ __forceinline__ float get(int j, bool in, int c, int n_ch) const { return in && c + j < n_ch ? A::to_float(r[j]) : 0.f; }
};

// 1 / (1 + e^-x) to two or three units in the last place, however small it is, in a third of the instructions that expf and a division
// take: the hardware's power of two and reciprocal, and what the rounding of the power's argument t left over, -x - t ln 2 (for x = -20
// it would move the gate by 1e-6 of itself).  NaN stays NaN; where x or t is infinite there is no rest.
__device__ __forceinline__ float sigmoid_gate(float x) {
  const float t = x * -1.4426950408889634f;
  const float rest = __builtin_fmaf(t, 1.9046543e-09f, __builtin_fmaf(t, -0.69314718246459961f, -x));
  return __builtin_amdgcn_rcpf(__builtin_fmaf(__builtin_amdgcn_exp2f(t), 1.0f + (fabsf(rest) < 1.0f ? rest : 0.f), 1.0f));
}

// A product of decays with what its roundings left over: the value is rounded once, however many factors it has.
struct Product {
  float hi = 1.f, lo = 0.f;
  __device__ __forceinline__ void by(float f) {
    const float p = hi * f;
    lo = __builtin_fmaf(lo, f, __builtin_fmaf(hi, f, -p));
    hi = p;
  }
  __device__ __forceinline__ float value() const { return hi + lo; }
  __device__ __forceinline__ float times(float x) const { return __builtin_fmaf(x, hi, x * lo); }
  __device__ __forceinline__ float rest(float x, float product) const { return __builtin_fmaf(x, hi, -product) + x * lo; }
};
struct PlainProduct {
  float v = 1.f;
  __device__ __forceinline__ void by(float f) { v *= f; }
  __device__ __forceinline__ float value() const { return v; }
  __device__ __forceinline__ float times(float x) const { return x * v; }
};

// the consumer's state: KT tiles of 16 key channels x this lane's value channel
template <int KT>
struct State {
  f32x4 S[KT];
  __device__ __forceinline__ void load(const float* slot, int K, int V, int col, int g, bool fresh) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int kk = 16 * kt + 4 * g + e;
        S[kt][e] = !fresh && col < V && kk < K ? slot[(int64_t)kk * V + col] : 0.f;
      }
  }
  __device__ __forceinline__ void store(float* slot, int K, int V, int col, int g) const {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int kk = 16 * kt + 4 * g + e;
        if (col < V && kk < K) slot[(int64_t)kk * V + col] = S[kt][e];
      }
  }
  // rows (token m) of x times the state; eight chains (shorter ones round less)
  __device__ __forceinline__ f32x4 times(const float* row) const {
    f32x4 o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(row + 16 * kt);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[4 * (kt & 1) + e] = mma4(x[e], S[kt][e], o[4 * (kt & 1) + e]);
    }
    return ((o[0] + o[1]) + (o[2] + o[3])) + ((o[4] + o[5]) + (o[6] + o[7]));
  }
};

// c plus a [16 x 16] matrix's rows (in LDS) times four accumulator rows
__device__ __forceinline__ f32x4 times_rows(const float* a, int m, int g, f32x4 w, f32x4 c = f32x4{0.f, 0.f, 0.f, 0.f}) {
  const f32x4 x = *reinterpret_cast<const f32x4*>(a + m * RA + 4 * g);
#pragma unroll
  for (int e = 0; e < 4; ++e) c = mma4(x[e], w[e], c);
  return c;
}

// The same summed in double (whose accumulator rows are 4 e + g where a float's are 4 g + e)
__device__ __forceinline__ f32x4 times_rows_double(const float* a, int m, int g, f32x4 w, f32x4 c) {
  const f32x4 x = *reinterpret_cast<const f32x4*>(a + row_of_token(m) * RA + 4 * g);
  f64x4 d = f64x4{c[0], c[1], c[2], c[3]};
#pragma unroll
  for (int e = 0; e < 4; ++e) d = __builtin_amdgcn_mfma_f64_16x16x4f64((double)x[e], (double)w[e], d, 0, 0, 0);
  return f32x4{(float)d[0], (float)d[1], (float)d[2], (float)d[3]};
}

// The same where a row of w may not be a finite number: nothing of it reaches the rows of tokens before its own (zero times infinity
// would).  Rare, and slow: on the vector ALU, a token after the other.
__device__ __forceinline__ f32x4 times_rows_in_order(const float* a, int m, int g, f32x4 w) {
  f32x4 c = f32x4{0.f, 0.f, 0.f, 0.f};
  asm volatile("" : "+v"(m), "+v"(g));                     // (nothing of this is worked out ahead of the loop over chunks)
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll 1
    for (int h = 0; h < 4; ++h) {                          // row 4 h + f, token 4 f + h
      const float x = __shfl(w[f], 16 * h + m, 64);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (4 * f + h <= 4 * e + g) c[e] = __builtin_fmaf(a[(4 * g + e) * RA + 4 * h + f], x, c[e]);
    }
  return c;
}
// uniform: some number of some lane is infinite or none
__device__ __forceinline__ bool some_not_finite(f32x4 w) {
  const bool fine = __builtin_isfinite(w[0]) && __builtin_isfinite(w[1]) && __builtin_isfinite(w[2]) && __builtin_isfinite(w[3]);
  return __builtin_amdgcn_ballot_w64(!fine) != 0;
}

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

// A chunk's rows on their way to LDS: NT threads, [16][W] of them, four channels a piece; row stride in LDS W + 4.
template <typename A, bool VEC, int W, int NT>
struct Rows {
  static constexpr int N = C * W / 4 / NT;
  Piece<A, 4, VEC> p[N];
  __device__ __forceinline__ static int row_of(int i, int tid) { return (tid + i * NT) / (W / 4); }
  __device__ __forceinline__ static int col_of(int i, int tid) { return (tid + i * NT) % (W / 4) * 4; }
  // base: channel 0 of the first token; n >= 1 tokens; channels c0 .. of n_ch
  __device__ __forceinline__ void fetch(const typename A::storage* base, int64_t stride, int c0, int n_ch, int n, int tid) {
#pragma unroll
    for (int i = 0; i < N; ++i) p[i].load(base + min(row_of(i, tid), n - 1) * stride, c0 + col_of(i, tid), n_ch);
  }
  __device__ __forceinline__ void store(float* lds, int c0, int n_ch, int n, float scale, int tid) const {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      f32x4 f;
#pragma unroll
      for (int j = 0; j < 4; ++j) f[j] = p[i].get(j, row_of(i, tid) < n, c0 + col_of(i, tid), n_ch) * scale;
      *reinterpret_cast<f32x4*>(lds + row_of_token(row_of(i, tid)) * (W + 4) + col_of(i, tid)) = f;
    }
  }
};

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
        w = times_rows(M, m, g, x);
      } else {
        const f32x4 s = *reinterpret_cast<const f32x4*>(sc + C + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = x[e] * s[e];
      }
      const f32x4 before = st.times(q);
      f32x4 within = times_rows(A, m, g, w);
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
// x[0 .. 31] of every lane: lane l ends with the sum over the wave of x[l / 2].  Every step keeps half of the values and adds
// the partner's share of them: 32 values in 75 instructions instead of 32 x 6.
template <int CTRL>
__device__ __forceinline__ float pair_sum(float keep, float give) { return keep + dpp_move<CTRL>(give); }
__device__ __forceinline__ float swap32_sum(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  const unsigned lo = r[0], hi = r[1];                    // (a bit cast of r[1] itself is taken from r[0] by this compiler)
  return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}
__device__ __forceinline__ float swap16_sum(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  const unsigned lo = r[0], hi = r[1];
  return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}
__device__ __forceinline__ float transpose_sum32(const float* x, int lane) {
  float y[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) y[i] = swap32_sum(x[i], x[i + 16]);      // (lanes 32 .. hold the second of the two)
#pragma unroll
  for (int i = 0; i < 8; ++i) y[i] = swap16_sum(y[i], y[i + 8]);
  const bool b8 = lane & 8, b4 = lane & 4, b2 = lane & 2;
#pragma unroll
  for (int i = 0; i < 4; ++i) y[i] = pair_sum<kDppMirror>(b8 ? y[i + 4] : y[i], b8 ? y[i] : y[i + 4]);
#pragma unroll
  for (int i = 0; i < 2; ++i) y[i] = pair_sum<kDppHalfMirror>(b4 ? y[i + 2] : y[i], b4 ? y[i] : y[i + 2]);
  y[0] = pair_sum<kDppXor2>(b2 ? y[1] : y[0], b2 ? y[0] : y[1]);
  return pair_sum<kDppXor1>(y[0], y[0]);
}
__device__ __forceinline__ float wave_total(float v) {
  v = row16_sum(v);
  v = swap16_sum(v, v);
  return swap32_sum(v, v);
}

template <int KP, int FORM, typename QK, typename VT, bool VEC>
__global__ __launch_bounds__(768) void chunk_channel_kernel(ChunkScanArgs a) {
  constexpr int KT = KP / 16, RS = KP + 4, NP = KP / 64;  // NP key channels a lane of a producer wave
  constexpr bool GATED = FORM == hxm::kChunkGated, BONUS = FORM == hxm::kChunkBonus;
  constexpr int kGate = C * KP * (GATED ? 2 : 3);         // decays | q | k
  // q times prefix | (k times suffix)^T | A | total | what the rounding of (k times suffix)^T left over, in bfloat16 (bonus form: its
  // k v is often exact, and a rounded factor would be the larger part of the state's error)
  constexpr int kMade = C * RS + KP * RA + C * RA + KP + (BONUS ? KP * RA / 2 : 0);
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
      f32x4 o = BONUS ? times_rows_double(A, m, g, w, before) : times_rows(A, m, g, w, before);
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

  // Producers, four waves that bring rows in and four that finish them: wave w (modulo 4) owns tokens 4 w .. 4 w + 3 of a chunk
  // (and their columns of A), lane l key channels NP l ..
  const int qk_head = GATED ? head : head / (a.heads / a.qk_heads);
  const int d0 = NP * lane;
  float u[NP], bias[NP], low[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const bool in = d0 + p < a.K;
    u[p] = BONUS && in ? a.bonus[(int64_t)head * a.K + d0 + p] : 0.f;
    bias[p] = GATED && in ? a.f_bias[(int64_t)head * a.K + d0 + p] : 0.f;
    low[p] = GATED && in ? a.low[(int64_t)head * a.K + d0 + p] : 0.f;
  }
  if (wave >= 8) {
    const int tid = (int)threadIdx.x - 512;
    struct Set {
      Piece<QK, NP, VEC> q[4], k[4];
      Piece<F32, NP, VEC> d[GATED ? 1 : 4];
      Rows<VT, VEC, VW, 256> values;
      float s;
    } sets[kAhead];
    const typename QK::storage* qp = (const typename QK::storage*)a.q + t_begin * a.q_stride + (int64_t)qk_head * a.K;
    const typename QK::storage* kp = (const typename QK::storage*)a.k + t_begin * a.k_stride + (int64_t)qk_head * a.K;
    const typename VT::storage* vp = (const typename VT::storage*)a.v + t_begin * a.v_stride + (int64_t)head * a.V;
    const int64_t d_stride = (int64_t)a.heads * a.K;
    const float* dp = GATED ? nullptr : a.decay + t_begin * d_stride + (int64_t)head * a.K;
    const float* sp = FORM == hxm::kChunkDecay ? (a.vscale ? a.vscale : a.decay) + t_begin * a.heads + head : nullptr;
    // (straight requests, kAhead chunks ahead; behind the last chunk the last one comes again)
    auto fetch = [&](Set& x, int chunk) __attribute__((always_inline)) {
      chunk = min(chunk, n_chunks - 1);
      const int n = rows_of(chunk);
      const int64_t t0 = (int64_t)chunk * C;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t t = t0 + min(4 * (wave - 8) + j, n - 1);
        x.q[j].load(qp + t * a.q_stride, d0, a.K);
        x.k[j].load(kp + t * a.k_stride, d0, a.K);
        if constexpr (!GATED) x.d[j].load(dp + t * d_stride, d0, a.K);
      }
      x.values.fetch(vp + t0 * a.v_stride, a.v_stride, col0, a.V, n, tid);
      if constexpr (FORM == hxm::kChunkDecay) x.s = sp[(t0 + min(x.values.row_of(0, tid), n - 1)) * a.heads];
    };
    auto store = [&](const Set& x, int chunk) __attribute__((always_inline)) {
      if (chunk >= n_chunks) return;
      const int n = rows_of(chunk);
      float* G = gates(chunk);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = 4 * (wave - 8) + j;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          const bool in = t < n && d0 + p < a.K;            // (a row past the portion, a channel past the key: nothing changes)
          const float qv = x.q[j].get(p, t < n, d0, a.K), kv = x.k[j].get(p, t < n, d0, a.K);
          if constexpr (GATED) {
            G[t * KP + d0 + p] = in ? low[p] + (1.0f - low[p]) * sigmoid_gate(kv + bias[p]) : 1.f;
            G[C * KP + t * KP + d0 + p] = qv * sigmoid_gate(qv);
          } else {
            G[t * KP + d0 + p] = in ? x.d[j].get(p, true, d0, a.K) : 1.f;
            G[C * KP + t * KP + d0 + p] = qv;
            G[2 * C * KP + t * KP + d0 + p] = kv;
          }
        }
      }
      x.values.store(vals(chunk), col0, a.V, n, FORM == hxm::kChunkDecay && a.vscale ? x.s : 1.f, tid);
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
  // Wave W makes columns W, 7 - W, 8 + W and 15 - W of A (34 elements each wave) and rows 4 W .. of the scaled q and k.  After the
  // butterfly lane l holds element l / 2 of the first 32: where it goes in A.
  int to;
  {
    const int W = wave, i = lane >> 1;
    int s, t;
    if (i < 16 - W) s = W, t = W + i;
    else if (i < 25) s = 7 - W, t = 7 - W + i - (16 - W);
    else if (i < 33 - W) s = 8 + W, t = 8 + W + i - 25;
    else s = 15 - W, t = 15 - W + i - (33 - W);
    to = row_of_token(t) * RA + row_of_token(s);
  }
  auto finish_wave = [&](int chunk, auto W_) __attribute__((always_inline)) {
    constexpr int W = decltype(W_)::value, S0 = 4 * W;
    constexpr int column[4] = {W, 7 - W, 8 + W, 15 - W};
    const float* G = gates(chunk);
    float* P = made(chunk);
    float* A = P + C * RS + KP * RA;
    float f[C][NP], q[C][NP];
#pragma unroll
    for (int t = 0; t < C; ++t)
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        f[t][p] = G[t * KP + d0 + p];
        q[t][p] = G[C * KP + t * KP + d0 + p];
      }
    float x[34];
    int at = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float run[NP];
#pragma unroll
      for (int p = 0; p < NP; ++p) run[p] = GATED ? 1.0f - f[column[j]][p] : G[2 * C * KP + column[j] * KP + d0 + p];
#pragma unroll
      for (int t = column[j]; t < C; ++t) {
        float s = 0.f;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          if (t > column[j] && !BONUS) run[p] *= f[t][p];
          if (BONUS && t == column[j]) s = __builtin_fmaf(q[t][p] * run[p], u[p], s);
          else s += q[t][p] * run[p];
          if (t > column[j] && BONUS) run[p] *= f[t][p];
        }
        x[at++] = s;
      }
    }
    // prefixes up to this wave's tokens, suffixes behind them (the gated form, whose decays are computed here, has no use for the
    // rest of a product: its state is off by less than before)
    typedef std::conditional_t<GATED, PlainProduct, Product> Decays;
    Decays pre[NP], suf[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
#pragma unroll
      for (int t = 0; t < S0; ++t) pre[p].by(f[t][p]);
#pragma unroll
      for (int t = C - 1; t >= S0 + 4; --t) suf[p].by(f[t][p]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        if (!BONUS) pre[p].by(f[S0 + j][p]);
        P[row_of_token(S0 + j) * RS + d0 + p] = pre[p].times(q[S0 + j][p]);
        if (BONUS) pre[p].by(f[S0 + j][p]);
      }
    if (W == 3) {
#pragma unroll
      for (int p = 0; p < NP; ++p) A[C * RA + d0 + p] = pre[p].value();
    }
#pragma unroll
    for (int j = 3; j >= 0; --j)
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const float k = GATED ? 1.0f - f[S0 + j][p] : G[2 * C * KP + (S0 + j) * KP + d0 + p], ks = suf[p].times(k);
        P[C * RS + (d0 + p) * RA + row_of_token(S0 + j)] = ks;
        if constexpr (BONUS) reinterpret_cast<u16*>(A + C * RA + KP)[(d0 + p) * RA + row_of_token(S0 + j)] = BF16::from_float(suf[p].rest(k, ks));
        if (j > 0) suf[p].by(f[S0 + j][p]);
      }
    // the last two elements by themselves: token 15 of columns 8 + W (W = 0) or 15 - W, and the one before it
    float last[2] = {wave_total(x[32]), wave_total(x[33])};
    const float sum = transpose_sum32(x, lane);
    if ((lane & 1) == 0) A[to] = sum;
    if (lane == 1) A[row_of_token(W == 0 ? 15 : 14) * RA + row_of_token(W == 0 ? 8 : 15 - W)] = last[0];
    if (lane == 3) A[row_of_token(15) * RA + row_of_token(15 - W)] = last[1];
  };
  auto finish = [&](int chunk) __attribute__((always_inline)) {
    if (chunk < 0 || chunk >= n_chunks) return;
    if (wave == 0) finish_wave(chunk, std::integral_constant<int, 0>());
    else if (wave == 1) finish_wave(chunk, std::integral_constant<int, 1>());
    else if (wave == 2) finish_wave(chunk, std::integral_constant<int, 2>());
    else finish_wave(chunk, std::integral_constant<int, 3>());
  };
  // the parts of A above its diagonal are never written again
  for (int i = threadIdx.x; i < C * RA; i += 256) {
    made(0)[C * RS + KP * RA + i] = 0.f;
    made(1)[C * RS + KP * RA + i] = 0.f;
  }
  for (int c = -2; c < n_chunks; ++c) {
    finish(c + 1);
    lds_barrier();
  }
}

template <typename Kernel>
int launch(Kernel kernel, int threads, size_t lds, const ChunkScanArgs& a, hipStream_t s) {
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
      hxm::last_hip_error() = (int)e;
      return HX_ERR_HIP;
    }
  }
  const dim3 grid((unsigned)a.heads, (unsigned)((a.V + VW - 1) / VW), (unsigned)a.n_seq);
  kernel<<<grid, dim3(threads), lds, s>>>(a);
  return hxm::check_launch();
}

template <int KP, typename QK, typename VT, bool VEC>
int launch_form(const ChunkScanArgs& a, hipStream_t s) {
  if (a.per_channel || a.form == hxm::kChunkGated) {
    const int kinds = a.form == hxm::kChunkGated ? 2 : 3;
    const size_t lds = sizeof(float) * (2 * C * KP * kinds + 2 * (C * (KP + 4) + KP * RA + C * RA + KP + (a.form == hxm::kChunkBonus ? KP * RA / 2 : 0)) + 3 * C * VS);
    if (a.form == hxm::kChunkGated) return launch(chunk_channel_kernel<KP, hxm::kChunkGated, QK, VT, VEC>, 768, lds, a, s);
    if (a.form == hxm::kChunkBonus) return launch(chunk_channel_kernel<KP, hxm::kChunkBonus, QK, VT, VEC>, 768, lds, a, s);
    return launch(chunk_channel_kernel<KP, hxm::kChunkDecay, QK, VT, VEC>, 768, lds, a, s);
  }
  const size_t lds = sizeof(float) * (3 * (2 * C * (KP + 4) + C * VS + 3 * C) + 2 * (2 * C * RA + 3 * C));
  if (a.form == hxm::kChunkDelta) return launch(chunk_head_kernel<KP, true, QK, VT, VEC>, 512, lds, a, s);
  return launch(chunk_head_kernel<KP, false, QK, VT, VEC>, 512, lds, a, s);
}

template <typename QK, typename VT>
int launch_width(const ChunkScanArgs& a, hipStream_t s) {
  auto by4 = [](const void* p, int dtype, int64_t stride, int n) {
    return n % 4 == 0 && stride % 4 == 0 && (uintptr_t)p % (dtype == HX_F32 ? 16 : 8) == 0;
  };
  const bool vec = by4(a.q, a.q_dtype, a.q_stride, a.K) && by4(a.k, a.k_dtype, a.k_stride, a.K) && by4(a.v, a.v_dtype, a.v_stride, a.V) &&
                   (!a.per_channel || by4(a.decay, HX_F32, 4, a.K));
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

int chunk_scan(const ChunkScanArgs& a, hipStream_t s) {
  if (a.q_dtype == HX_BF16) return launch_width<BF16, BF16>(a, s);
  return a.v_dtype == HX_F32 ? launch_width<F32, F32>(a, s) : launch_width<F32, BF16>(a, s);
}

}  // namespace hxm
