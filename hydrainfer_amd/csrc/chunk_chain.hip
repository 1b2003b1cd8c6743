// chunk_chain.hip — the recurrences with a decay per key channel over portions of prompts, sixteen tokens at a time (chunk_scan.hip says
// how), in two launches: what does not depend on the state — A, the prefixed queries, the suffixed keys, all of it vector work — is
// made for all chunks at once on the whole chip, and the chain of chunks is left with the products of the state.  One launch has these
// made beside the chain, on the same SIMDs and once per 64 value channels: a chunk of the gated form with 128 x 128 took 2.6 us there and
// takes 1.5 here, of which 0.95 are the products.  (Vector instructions of a consumer's own wave do not run beside its float products: a
// multiplication behind each of them costs 7 cycles of 32; those of other waves cost nothing.  So results leave through LDS by the
// waves that bring rows in.)  Measured, gated form, one launch and two with the norm: 4 portions of 797 - 1151 tokens, 32 heads of 128 x
// 128 206 and 176 us; one of 1151, 4 heads 189 and 115, 64 x 64 117 and 72.  The first launch takes 53 us of the 176 (vector work: 560
// instructions a wave of four tokens; 164 MB written), and so what it costs is weighed against the chain (chunk_scan_workspace).
// Head-wise decays gain too little: with A and M made ahead the chain of the delta rule is bound by its own waves (2.5 -> 2.3 us a
// chunk, 104 products of 32 cycles and 140 vector instructions of 7), and the launch ahead takes what it gives (204 and 199 us).
#include "chunk_parts.h"

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

// A chunk's results [16][VW] on their way from LDS, where they stand by row, to memory: 256 threads, four channels each.
template <bool VEC>
__device__ __forceinline__ void write_results(const ChunkScanArgs& a, const float* lds, int64_t t0, int n, int head, int col0, int tid) {
  const int t = tid / (VW / 4), col = col0 + tid % (VW / 4) * 4;
  const f32x4 o = *reinterpret_cast<const f32x4*>(lds + row_of_token(t) * VS + tid % (VW / 4) * 4);
  float* to = a.out + (t0 + t) * ((int64_t)a.heads * a.V) + (int64_t)head * a.V + col;
  if (t >= n) return;
  if (VEC) {
    if (col < a.V) *reinterpret_cast<f32x4*>(to) = o;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col + e < a.V) to[e] = o[e];
  }
}

// What the chunks need besides their values, all chunks at once.
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

template <int KP, int FORM, typename VT, bool VEC>
__global__ __launch_bounds__(512, KP == 64 ? 4 : 2) void chunk_channel_chain_kernel(ChunkScanArgs a) {
  constexpr int KT = KP / 16, RS = KP + 4;
  constexpr bool BONUS = FORM == hxm::kChunkBonus;
  constexpr int kMade = kMadeChannel<KP, FORM>;
  extern __shared__ __attribute__((aligned(16))) float lds[];      // made[2] | values[2] | results[2]
  const int seq = blockIdx.z, head = blockIdx.x, col0 = (int)blockIdx.y * VW;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, m = lane & 15;
  const int64_t t_begin = a.q_cu[seq];
  const int n_tok = (int)(a.q_cu[seq + 1] - t_begin);
  if (n_tok <= 0) return;                                 // (the whole workgroup)
  const int n_chunks = (n_tok + C - 1) / C;
  float* slot = a.state + (int64_t)a.slots[seq] * a.slot_stride + (int64_t)head * a.K * a.V;
  auto made = [&](int chunk) { return lds + (chunk & 1) * kMade; };
  auto vals = [&](int chunk) { return lds + 2 * kMade + (chunk & 1) * (C * VS); };
  auto outs = [&](int chunk) { return lds + 2 * kMade + (2 + (chunk & 1)) * (C * VS); };
  auto rows_of = [&](int chunk) { return min(C, n_tok - chunk * C); };

  if (wave >= 4) {
    const int cw = wave - 4, col = col0 + 16 * cw + m;
    State<KT> st;
    st.load(slot, a.K, a.V, col, g, a.positions[t_begin] == 0);
    lds_barrier();
    // What a chunk's first products take is read behind the barrier that ends the chunk before, whose products with its keys follow it.
    f32x4 qx[KT];
    read_row(qx, made(0) + m * RS + 4 * g);
    for (int c = 0; c < n_chunks; ++c) {
      const float* p = made(c);
      const float *kt_ = p + C * RS, *A = kt_ + KP * RA, *total = A + C * RA;
      const float* vs = vals(c) + 4 * g * VS + 16 * cw + m;
      f32x4 w, kx[KT], d[KT];
      s16x4 w16, ky[KT];
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = vs[e * VS];
      const f32x4 A_row = *reinterpret_cast<const f32x4*>(A + (BONUS ? row_of_token(m) : m) * RA + 4 * g);
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        d[kt] = *reinterpret_cast<const f32x4*>(total + 16 * kt + 4 * g);
        kx[kt] = *reinterpret_cast<const f32x4*>(kt_ + (16 * kt + m) * RA + 4 * g);
        if constexpr (BONUS) ky[kt] = *reinterpret_cast<const s16x4*>(reinterpret_cast<const u16*>(total + KP) + (16 * kt + m) * RA + 4 * g);
      }
      const f32x4 before = st.times(qx);
      __builtin_amdgcn_sched_group_barrier(0x100, 64, 0);
      const bool odd = some_not_finite(w);
      f32x4 in_order = f32x4{0.f, 0.f, 0.f, 0.f};
      if (odd) in_order = times_rows_in_order(A, m, g, w);
      lds_barrier();
      read_row(qx, made(c + 1) + m * RS + 4 * g);         // (behind the last chunk: the one before it, unused)
#pragma unroll
      for (int e = 0; e < 4; ++e) w16[e] = (short)BF16::from_float(w[e]);
      f32x4 o = BONUS ? times_rows_double(A_row, w, before) : times_rows(A_row, w, before);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = odd ? before[e] + in_order[e] : o[e];
#pragma unroll
      for (int e = 0; e < 4; ++e) outs(c)[(4 * g + e) * VS + 16 * cw + m] = o[e];
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        if constexpr (BONUS) {
          const f32x4 rest = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ky[kt], w16, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) st.S[kt][e] = __builtin_fmaf(st.S[kt][e], d[kt][e], rest[e]);
        } else {
          st.S[kt] *= d[kt];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) st.S[kt] = mma4(kx[kt][e], w[e], st.S[kt]);
      }
    }
    lds_barrier();
    st.store(slot, a.K, a.V, col, g);
    return;
  }

  const typename VT::storage* vp = (const typename VT::storage*)a.v + t_begin * a.v_stride + (int64_t)head * a.V;
  const float* sp = FORM == hxm::kChunkDecay ? (a.vscale ? a.vscale : a.decay) + t_begin * a.heads + head : nullptr;
  // Four waves that bring in the values and what was made of the keys and queries, kAhead chunks ahead of the interval that puts them in
  // LDS: an interval is shorter than a load's way.  Behind the last chunk the last one comes again.
  const int tid = (int)threadIdx.x;
  const float* from = a.made + (chunk_number(t_begin, seq) * a.heads + head) * kMade;
  struct Set {
    MadeRows<kMade, 256> made;
    Rows<VT, VEC, VW, 256> v;
    float scale;
  } sets[kAhead];
  auto fetch = [&](Set& s, int chunk) __attribute__((always_inline)) {
    chunk = min(chunk, n_chunks - 1);
    const int n = rows_of(chunk);
    const int64_t t0 = (int64_t)chunk * C;
    s.made.fetch(from + (int64_t)chunk * a.heads * kMade, tid);
    s.v.fetch(vp + t0 * a.v_stride, a.v_stride, col0, a.V, n, tid);
    if constexpr (FORM == hxm::kChunkDecay) s.scale = sp[(t0 + min(s.v.row_of(0, tid), n - 1)) * a.heads];
  };
  auto store = [&](const Set& s, int chunk) __attribute__((always_inline)) {
    if (chunk >= n_chunks) return;
    s.made.store(made(chunk), tid);
    s.v.store(vals(chunk), col0, a.V, rows_of(chunk), FORM == hxm::kChunkDecay && a.vscale ? s.scale : 1.f, tid);
  };
#pragma unroll
  for (int i = 0; i < kAhead; ++i) fetch(sets[i], i);
  for (int c0 = -1; c0 < n_chunks; c0 += kAhead) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int c = c0 + i;
      if (c >= n_chunks) break;
      store(sets[i], c + 1);
      fetch(sets[i], c + 1 + kAhead);
      if (c >= 2) write_results<VEC>(a, outs(c - 2), t_begin + (int64_t)(c - 2) * C, C, head, col0, tid);      // (chunk c - 1's are being written)
      lds_barrier();
    }
  }
  if (n_chunks >= 2) write_results<VEC>(a, outs(n_chunks - 2), t_begin + (int64_t)(n_chunks - 2) * C, C, head, col0, tid);
  lds_barrier();
  write_results<VEC>(a, outs(n_chunks - 1), t_begin + (int64_t)(n_chunks - 1) * C, rows_of(n_chunks - 1), head, col0, tid);
}

// numbers that chunks may have
int64_t chunk_numbers(const ChunkScanArgs& a) { return a.n_tokens / C + a.n_seq; }
template <int KP>
int64_t made_floats(const ChunkScanArgs& a) {
  return a.form == hxm::kChunkGated ? kMadeChannel<KP, hxm::kChunkGated> : a.form == hxm::kChunkBonus ? kMadeChannel<KP, hxm::kChunkBonus> : kMadeChannel<KP, hxm::kChunkDecay>;
}

template <int KP, int FORM, typename QK, typename VT, bool VEC>
int launch_channel(const ChunkScanArgs& a, hipStream_t s) {
  const int rc = launch_chunks(chunk_channel_make_kernel<KP, FORM, QK, VEC>, dim3((unsigned)(chunk_numbers(a) * a.heads)), 256, 0, a, s);
  if (rc != HX_OK) return rc;
  return launch_chunks(chunk_channel_chain_kernel<KP, FORM, VT, VEC>, dim3((unsigned)a.heads, (unsigned)((a.V + VW - 1) / VW), (unsigned)a.n_seq), 512,
                       sizeof(float) * (2 * kMadeChannel<KP, FORM> + 4 * C * VS), a, s);
}

template <int KP, typename QK, typename VT, bool VEC>
int launch_form(const ChunkScanArgs& a, hipStream_t s) {
  if (a.form == hxm::kChunkGated) return launch_channel<KP, hxm::kChunkGated, QK, VT, VEC>(a, s);
  if (a.form == hxm::kChunkBonus) return launch_channel<KP, hxm::kChunkBonus, QK, VT, VEC>(a, s);
  return launch_channel<KP, hxm::kChunkDecay, QK, VT, VEC>(a, s);
}

template <typename QK, typename VT>
int launch_width(const ChunkScanArgs& a, hipStream_t s) {
  const bool vec = rows_by_four(a) && (uintptr_t)a.out % 16 == 0;
  if (a.K <= 64) return vec ? launch_form<64, QK, VT, true>(a, s) : launch_form<64, QK, VT, false>(a, s);
  return vec ? launch_form<128, QK, VT, true>(a, s) : launch_form<128, QK, VT, false>(a, s);
}

}  // namespace

namespace hxm {

int64_t chunk_scan_workspace(const ChunkScanArgs& a) {
  if (!chunk_scan_fits(a) || !(a.per_channel || a.form == kChunkGated)) return 0;
  const int64_t workgroups = chunk_numbers(a) * a.heads;
  const int64_t floats = workgroups * (a.K <= 64 ? made_floats<64>(a) : made_floats<128>(a));
  if (workgroups > INT32_MAX || floats > (int64_t)1 << 28) return 0;      // (1 GiB)
  // Two launches save `gain` us for a chunk of the chain and take `cost` us for each chunk and head, and 2 us.  Fitted to batches of 1 to
  // 64 portions of 32 to 1151 tokens and 4 to 32 heads, one launch and two, us: gated form, 128 x 128, 32 heads: 1 of 1151 197 131, 4 of
  // 1000 189 175, 4 of 128 34 34, 4 of 64 21 24; 64 x 64: 1 of 1151 121 84, 4 of 128 22 24, 8 of 512 68 77; bonus form, 64 x 64, 32 heads: 1 of
  // 1151 109 95, 4 of 1000 100 105, 8 heads: 4 of 256 29 28, of 64 11 14; 128 x 128, 32 heads: 4 of 256 50 56, 16 heads 48 47; a decay per
  // channel, 128 x 64, 32 heads: 4 of 256 44 47, 16 heads 43 41, 8 of 512 85 124.
  const bool wide = a.K > 64;
  const double gain = a.form == kChunkGated ? (wide ? 1.0 : 0.6) : a.form == kChunkBonus ? (wide ? 0.6 : 0.28) : wide ? 0.7 : 0.28, cost = wide ? 0.0067 : 0.0025;
  const double mean = (double)a.n_tokens / a.n_seq / C, longest = a.longest > 0 ? (double)a.longest / C : mean;
  const int64_t chains = (int64_t)a.n_seq * a.heads * ((a.V + VW - 1) / VW);      // a compute unit takes one at a time
  return gain * (chains <= 256 ? longest : mean * ((chains + 255) / 256)) > cost * a.n_tokens / C * a.heads + 3.0 ? floats : 0;
}

int chunk_chain(const ChunkScanArgs& a, hipStream_t s) {
  if (a.q_dtype == HX_BF16) return launch_width<BF16, BF16>(a, s);
  return a.v_dtype == HX_F32 ? launch_width<F32, F32>(a, s) : launch_width<F32, BF16>(a, s);
}

}  // namespace hxm
