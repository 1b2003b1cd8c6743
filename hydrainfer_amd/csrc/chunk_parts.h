// chunk_parts.h — what the two forms of the recurrences over portions of prompts share (chunk_scan.hip: one launch; chunk_chain.hip: what
// the chunks need made in a launch ahead): operands on their way, products with the state, and the matrices of a chunk.
#pragma once
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

// this lane's part of a row of operands, sixteen channels apart
template <int KT>
__device__ __forceinline__ void read_row(f32x4 (&x)[KT], const float* row) {
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) x[kt] = *reinterpret_cast<const f32x4*>(row + 16 * kt);
}

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
  __device__ __forceinline__ f32x4 times(const f32x4 (&x)[KT]) const {
    f32x4 o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) o[4 * (kt & 1) + e] = mma4(x[kt][e], S[kt][e], o[4 * (kt & 1) + e]);
    return ((o[0] + o[1]) + (o[2] + o[3])) + ((o[4] + o[5]) + (o[6] + o[7]));
  }
  __device__ __forceinline__ f32x4 times(const float* row) const {
    f32x4 x[KT];
    read_row(x, row);
    return times(x);
  }
};

// c plus a [16 x 16] matrix's rows (x: this lane's four numbers of row m) times four accumulator rows
__device__ __forceinline__ f32x4 times_rows(f32x4 x, f32x4 w, f32x4 c = f32x4{0.f, 0.f, 0.f, 0.f}) {
#pragma unroll
  for (int e = 0; e < 4; ++e) c = mma4(x[e], w[e], c);
  return c;
}

// The same summed in double (whose accumulator rows are 4 e + g where a float's are 4 g + e)
__device__ __forceinline__ f32x4 times_rows_double(f32x4 x, f32x4 w, f32x4 c) {
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
// One decay per token and key channel.
// ---------------------------------------------------------------------------------------------------------------
// Sixteen tokens' decays | q | k (gated form: 1 - decay), and what is made of them for a chunk: q times prefix | (k times suffix)^T | A |
// total | what the rounding of (k times suffix)^T left over, in bfloat16 (bonus form: its k v is often exact, and a rounded factor
// would be the larger part of the state's error)
template <int KP, int FORM>
constexpr int kGateFloats = C * KP * (FORM == hxm::kChunkGated ? 2 : 3);
template <int KP, int FORM>
constexpr int kMadeChannel = C * (KP + 4) + KP * RA + C * RA + KP + (FORM == hxm::kChunkBonus ? KP * RA / 2 : 0);

// a lane's key channels' own numbers
template <int NP, int FORM>
struct ChannelBias {
  float u[NP], bias[NP], low[NP];
  __device__ __forceinline__ ChannelBias(const ChunkScanArgs& a, int head, int d0) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const bool in = d0 + p < a.K;
      u[p] = FORM == hxm::kChunkBonus && in ? a.bonus[(int64_t)head * a.K + d0 + p] : 0.f;
      bias[p] = FORM == hxm::kChunkGated && in ? a.f_bias[(int64_t)head * a.K + d0 + p] : 0.f;
      low[p] = FORM == hxm::kChunkGated && in ? a.low[(int64_t)head * a.K + d0 + p] : 0.f;
    }
  }
};

// Rows of a chunk on their way to LDS: wave W (of four) tokens 4 W .. 4 W + 3, lane l key channels NP l ..
template <int KP, int FORM, typename QK, bool VEC>
struct GateRows {
  static constexpr int NP = KP / 64;
  static constexpr bool GATED = FORM == hxm::kChunkGated;
  Piece<QK, NP, VEC> q[4], k[4];
  Piece<F32, NP, VEC> d[GATED ? 1 : 4];
  // q0, k0, dec0: the head's channel 0 of the chunk's first token
  __device__ __forceinline__ void fetch(const typename QK::storage* q0, int64_t q_stride, const typename QK::storage* k0, int64_t k_stride, const float* dec0, int64_t d_stride,
                                        int n, int K, int W, int d0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t t = min(4 * W + j, n - 1);
      q[j].load(q0 + t * q_stride, d0, K);
      k[j].load(k0 + t * k_stride, d0, K);
      if constexpr (!GATED) d[j].load(dec0 + t * d_stride, d0, K);
    }
  }
  __device__ __forceinline__ void store(float* G, const ChannelBias<NP, FORM>& own, int n, int K, int W, int d0) const {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = 4 * W + j;
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const bool in = t < n && d0 + p < K;                // (a row past the portion, a channel past the key: nothing changes)
        const float qv = q[j].get(p, t < n, d0, K), kv = k[j].get(p, t < n, d0, K);
        if constexpr (GATED) {
          float f = own.low[p] + (1.0f - own.low[p]) * sigmoid_gate(kv + own.bias[p]);
          asm("" : "+v"(f));                                // (no branch around it: it would stand between every two elements)
          G[t * KP + d0 + p] = in ? f : 1.f;
          G[C * KP + t * KP + d0 + p] = qv * sigmoid_gate(qv);
        } else {
          G[t * KP + d0 + p] = in ? d[j].get(p, true, d0, K) : 1.f;
          G[C * KP + t * KP + d0 + p] = qv;
          G[2 * C * KP + t * KP + d0 + p] = kv;
        }
      }
    }
  }
};

// Wave W makes columns W, 7 - W, 8 + W and 15 - W of A (34 elements each wave) and rows 4 W .. of the scaled q and k.  After the
// butterfly lane l holds element l / 2 of the first 32: where it goes in A.
__device__ __forceinline__ int place_in_A(int W, int lane) {
  const int i = lane >> 1;
  int s, t;
  if (i < 16 - W) s = W, t = W + i;
  else if (i < 25) s = 7 - W, t = 7 - W + i - (16 - W);
  else if (i < 33 - W) s = 8 + W, t = 8 + W + i - 25;
  else s = 15 - W, t = 15 - W + i - (33 - W);
  return row_of_token(t) * RA + row_of_token(s);
}
template <int KP, int FORM, int W>
__device__ __forceinline__ void finish_rows(const float* G, float* P, const ChannelBias<KP / 64, FORM>& own, int to, int lane) {
  constexpr int NP = KP / 64, RS = KP + 4, S0 = 4 * W;
  constexpr bool GATED = FORM == hxm::kChunkGated, BONUS = FORM == hxm::kChunkBonus;
  constexpr int column[4] = {W, 7 - W, 8 + W, 15 - W};
  const int d0 = NP * lane;
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
        if (BONUS && t == column[j]) s = __builtin_fmaf(q[t][p] * run[p], own.u[p], s);
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
}
template <int KP, int FORM>
__device__ __forceinline__ void finish_chunk(const float* G, float* P, const ChannelBias<KP / 64, FORM>& own, int to, int wave, int lane) {
  if (wave == 0) finish_rows<KP, FORM, 0>(G, P, own, to, lane);
  else if (wave == 1) finish_rows<KP, FORM, 1>(G, P, own, to, lane);
  else if (wave == 2) finish_rows<KP, FORM, 2>(G, P, own, to, lane);
  else finish_rows<KP, FORM, 3>(G, P, own, to, lane);
}

// Rows of four channels at a time: n, the stride and the pointer allow it.
inline bool rows_by_four(const ChunkScanArgs& a) {
  auto by4 = [](const void* p, int dtype, int64_t stride, int n) {
    return n % 4 == 0 && stride % 4 == 0 && (uintptr_t)p % (dtype == HX_F32 ? 16 : 8) == 0;
  };
  return by4(a.q, a.q_dtype, a.q_stride, a.K) && by4(a.k, a.k_dtype, a.k_stride, a.K) && by4(a.v, a.v_dtype, a.v_stride, a.V) &&
         (!a.per_channel || by4(a.decay, HX_F32, 4, a.K));
}

template <typename Kernel>
int launch_chunks(Kernel kernel, dim3 grid, int threads, size_t lds, const ChunkScanArgs& a, hipStream_t s) {
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
      hxm::last_hip_error() = (int)e;
      return HX_ERR_HIP;
    }
  }
  kernel<<<grid, dim3(threads), lds, s>>>(a);
  return hxm::check_launch();
}

}  // namespace
