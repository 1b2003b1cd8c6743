// chunk_head.hip — recurrences with one decay per token and head over portions of prompts (chunk_scan.hip says how; the delta rule and the
// decayed sum), in one launch, thirty-two tokens at a time.  A chunk is two tiles of sixteen tokens:
//     W_0 = M_00 b (V - R)_0,  W_1 = M_11 b (V - R - T_10 W_0)_1      R = prefix (K S), M_uu = (I + b T_uu)^-1      (decayed sum: W = s V)
//     O_u = prefix (Q S) + sum(v <= u) A_uv W_v,  S <- total S + (K * suffix)^T W
// The products with the state and q k^T, k k^T are bfloat16 products of operands that are split in three (Henry, Tang and Heinecke, Leveraging the
// bfloat16 artificial intelligence datatype for higher-precision computations, 2019): x = hi + mid + lo, each rounded to bfloat16, holds all of a
// float's 24 bits, and of the nine products of two such numbers the three that are left out are below 2^-24 of the whole.  Six products of 16 x 16 x 32 take 96 cycles where float products of the same size take 256, and round less: hi hi is
// summed by itself and the other five beside it (2-norm of the error over 128 channels, operands normal: 8.8e-8 in float with eight
// chains, 6.5e-8 here; all six in one sum 1.5e-7).  bfloat16 q and k are one part and take three products, all of them exact.
// W, M, A and T stay float, and so do the state and everything that is added up.  Limits: lo is below bfloat16's smallest numbers where x is below
// 2^-110 (its parts are then off by up to 2^-134: subnormal ones are kept), and a finite x above 3.39e38 rounds to an infinite hi and counts as infinite.
// A workgroup owns 64 value channels of one (sequence, head): four consumer waves hold the state, 16 channels of values and all keys
// each, as accumulators, and split it anew for each chunk; the parts are the operand of the products with S as they lie in the registers
// (a lane group's eight keys: rows 4 g + e of two tiles of 16).  Four producer waves bring rows in (requested a chunk ahead), split
// them into planes in LDS and make A, M and T of the next chunk while the consumers work on this one; two barriers a chunk.
// What bounds it: the vector ALU of a SIMD, which a consumer (430 instructions a chunk under the delta rule: parts, sums, results) and a producer (850:
// parts of rows, products of decays, the substitution) share, and which does not run beside the products of its own wave.  Of a chunk's 4.6 us
// 1.3 are matrix products.
// Rows are read eight bytes at a time (two reads made one by the compiler bring a quarter of their bytes a cycle) and straight from global memory (through flat
// addresses every barrier waited for them): delta rule, 128 x 128, 32 heads, 4 portions of 797 - 1151 tokens 167.2 -> 159.2 us, the same bits.
// Measured before that, one launch of sixteen tokens at a time in float and this one, us: delta rule, 128 x 128, 32 heads, 4 portions of 797 - 1151 tokens 191 and
// 169, 12 of 300 - 900 348 and 309, 16 of 60 55.6 and 55.6; decayed sum, 128 x 128, 32 heads, 4 of 797 - 1151 145 and 103, 12 of 300 - 900 263 and 190,
// one of 100 19.8 and 17.1, 64 x 64 93 and 83.  Results' error against 64 bits (2-norm, 400 and 250 tokens, 1e-7): delta rule 1.08 and 1.00,
// decayed sum 128 x 128 0.867 and 0.863, 64 x 64 0.79 and 0.76; states 0.77 and 0.72, 0.73 and 0.62, 0.72 and 0.64.
#include <cfloat>

#include "attn_common.h"
#include "chunk_parts.h"

namespace {

constexpr int CW = 2 * C;          // tokens a chunk
constexpr int RM = CW + 4;         // floats a row of A, and of M with T

// Row of a token in the accumulators and in LDS: tiles of sixteen, each as row_of_token has it.
__device__ __forceinline__ constexpr int row_of(int t) { return (t & C) | row_of_token(t & (C - 1)); }
// Where a row of a tile lies in the planes: rows of 272 bytes start four banks apart, so that sixteen of them are read 16 bytes at a time without a
// conflict; the eight rows that a transposing read takes at once, 32 bytes each, are every other one.
__device__ __forceinline__ constexpr int place_of(int r) { return (r & C) | (r & 7) << 1 | (r >> 3 & 1); }

__device__ __forceinline__ f32x4 mma_parts(u16x8 a, u16x8 b, f32x4 c) {
  typedef __bf16 part_t __attribute__((ext_vector_type(8)));
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(part_t, a), __builtin_bit_cast(part_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ u16x8 both(u16x4 a, u16x4 b) { return u16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]}; }

// Four floats in three parts, two at a time: one conversion makes both numbers' parts.  (v_dot2_f32_bf16 would take a part from its float in one instruction and not in
// two: the delta rule on 4 portions of 797 - 1151 tokens, 32 heads of 128 x 128, 164 us and not 159, and states off by 5 % more, 7.12 and 7.44e-8.)
__device__ __forceinline__ void split(f32x4 x, u16x4 (&part)[3]) {
  typedef __bf16 pair_t __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int e = 0; e < 4; e += 2) {
      const uint32_t bits = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x[e], x[e + 1]}), pair_t));
      part[p][e] = (u16)bits;
      part[p][e + 1] = (u16)(bits >> 16);
      if (p < 2) {
        x[e] -= __builtin_bit_cast(float, bits << 16);
        x[e + 1] -= __builtin_bit_cast(float, bits & 0xffff0000u);
      }
    }
}

// What is infinite has no lower parts (inf - inf), and an infinity times another's lower part of zero is no number: where the sum of hi hi is not finite it
// says by itself what a product is, and the other sum, whatever it came to, is only to be finite.  (v_med3 with an operand that is no number gives the least of
// the others.)
__device__ __forceinline__ f32x4 total_of(const f32x4 (&sum)[2]) {
  f32x4 t;
#pragma unroll
  for (int e = 0; e < 4; ++e) t[e] = sum[0][e] + __builtin_amdgcn_fmed3f(sum[1][e], -FLT_MAX, FLT_MAX);
  return t;
}

// Products of N operands in parts with one in parts (SECOND: the other way round): hi hi to sum[0], the others, smallest first, to sum[1].  A product
// a turn of every operand: one waits for the one before it on the same sum.
template <bool SECOND = false, int N, int NA, int NB>
__device__ __forceinline__ void add_products(const u16x8 (&a)[N][NA], const u16x8 (&b)[NB], f32x4 (&sum)[N][2]) {
#pragma unroll
  for (int order = 2; order >= 0; --order)
#pragma unroll
    for (int i = NA - 1; i >= 0; --i)
#pragma unroll
      for (int n = 0; n < N; ++n)
        if (order - i >= 0 && order - i < NB)
          sum[n][order > 0] = SECOND ? mma_parts(b[order - i], a[n][i], sum[n][order > 0]) : mma_parts(a[n][i], b[order - i], sum[n][order > 0]);
}

// bytes of a chunk in LDS: planes of q and of k, values, A, M with T, numbers a token by row (value scale or write strength, prefix, what
// the prefix's rounding left over, suffix)
template <int KP, typename QK, bool DELTA>
struct HeadImage {
  static constexpr int NP = QK::kDtype == HX_BF16 ? 1 : 3;
  static constexpr int kRow = 2 * KP + 16, kPlane = CW * kRow;      // (16 rows that an instruction reads start in different banks)
  static constexpr int kQ = 0, kK = NP * kPlane, kV = 2 * NP * kPlane, kA = kV + 4 * CW * VS, kM = kA + 4 * CW * RM, kBytes = kM + (DELTA ? 4 * CW * RM : 0);
  // behind the two images, three chunks of them: they are made a chunk ahead
  static constexpr int kScale = 0, kPrefix = kScale + 4 * CW, kRest = kPrefix + 4 * CW, kSuffix = kRest + 4 * CW, kTokens = kSuffix + 4 * CW;
  static constexpr int kLds = 2 * kBytes + 3 * kTokens;
};

// sum over s <= t of a row's numbers times w's rows, where a row of w may not be a finite number (times_rows_in_order, rows RM floats apart)
__device__ __forceinline__ f32x4 rows_in_order(const float* a, int m, int g, f32x4 w, f32x4 c) {
  asm volatile("" : "+v"(m), "+v"(g));
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll 1
    for (int h = 0; h < 4; ++h) {
      const float x = __shfl(w[f], 16 * h + m, 64);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (4 * f + h <= 4 * e + g) c[e] = __builtin_fmaf(a[(4 * g + e) * RM + 4 * h + f], x, c[e]);
    }
  return c;
}

__device__ __forceinline__ Product product_of(const Product& a, const Product& b) {
  Product r;
  r.hi = a.hi * b.hi;
  r.lo = __builtin_fmaf(a.hi, b.hi, -r.hi) + __builtin_fmaf(a.hi, b.lo, a.lo * b.hi);
  return r;
}

template <int KP, bool DELTA, typename QK, typename VT, bool VEC>
__global__ __launch_bounds__(512) void chunk_head32_kernel(ChunkScanArgs a) {
  typedef HeadImage<KP, QK, DELTA> I;
  constexpr int KT = KP / 16, KB = KP / 32, NP = I::NP;
  extern __shared__ __attribute__((aligned(16))) char smem[];      // [2] images
  const int seq = blockIdx.z, head = blockIdx.x, col0 = (int)blockIdx.y * VW;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, m = lane & 15;
  const int64_t t_begin = a.q_cu[seq];
  const int n_tok = (int)(a.q_cu[seq + 1] - t_begin);
  if (n_tok <= 0) return;                                 // (the whole workgroup)
  const int n_chunks = (n_tok + CW - 1) / CW;
  auto image = [&](int chunk) { return smem + (chunk & 1) * I::kBytes; };
  auto tokens = [&](int chunk) { return smem + 2 * I::kBytes + chunk % 3 * I::kTokens; };
  auto rows_of = [&](int chunk) { return min(CW, n_tok - chunk * CW); };
  // 16 rows (row m of tile u) times 32 channels of an operand in parts; as A and as B operand alike
  // (two reads of eight bytes from addresses that the compiler does not know to be near each other: it would make one ds_read2_b64 of them, which
  // brings 64 bytes a cycle where the two bring 230)
  int half_at[2] = {place_of(m) * I::kRow + 8 * g, place_of(m) * I::kRow + 8 * g + 32};
  asm volatile("" : "+v"(half_at[1]));
  auto parts_at = [&](const char* planes, int u, int kb, u16x8 (&x)[NP]) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int at = p * I::kPlane + 16 * u * I::kRow + 64 * kb;
      x[p] = both(*reinterpret_cast<const u16x4*>(planes + half_at[0] + at), *reinterpret_cast<const u16x4*>(planes + half_at[1] + at));
    }
  };

  if (wave >= 4) {
    const int cw = wave - 4, col = col0 + 16 * cw + m;
    float* slot = a.state + (int64_t)a.slots[seq] * a.slot_stride + (int64_t)head * a.K * a.V;
    State<KT> st;
    st.load(slot, a.K, a.V, col, g, a.positions[t_begin] == 0);
    const int64_t out_row = (int64_t)a.heads * a.V;
    float* out = a.out + (t_begin + g) * out_row + (int64_t)head * a.V + col;      // (advanced by a chunk's rows)
    lds_barrier();                                        // chunk 0's rows are there
    for (int c = 0; c < n_chunks; ++c) {
      lds_barrier();                                      // what is made of them, too
      const char* im = image(c);
      // Products with the state: rows of q (and k) of both tiles, those of the next 32 channels on their way and the state's next parts made
      // under the products of these.
      constexpr int NX = DELTA ? 4 : 2;                   // q of both tiles, k of both
      f32x4 sum[NX][2];
#pragma unroll
      for (int i = 0; i < NX; ++i) sum[i][0] = sum[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
      u16x8 rows[2][NX][NP], sp[2][3];
      auto rows_at = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NX; ++i) parts_at(im + (i < 2 ? I::kQ : I::kK), i & 1, kb, rows[kb & 1][i]);
      };
      auto state_at = [&](int kb) __attribute__((always_inline)) {
        u16x4 s0[3], s1[3];
        split(st.S[2 * kb], s0);
        split(st.S[2 * kb + 1], s1);
#pragma unroll
        for (int p = 0; p < 3; ++p) sp[kb & 1][p] = both(s0[p], s1[p]);
      };
      // what the rest takes from LDS, asked for under the last of these products
      const char* tk = tokens(c);
      const float* A = reinterpret_cast<const float*>(im + I::kA);
      const float* M = reinterpret_cast<const float*>(im + I::kM);
      const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
      f32x4 w[2], scale[2], pre[2], rest[2], suffix[2], m00, m11, t10, a00, a10, a11;
      float total;
      auto token = [&](int what, int u) __attribute__((always_inline)) { return *reinterpret_cast<const f32x4*>(tk + what + 4 * (16 * u + 4 * g)); };
      auto row = [&](const float* of, int u, int v) __attribute__((always_inline)) { return *reinterpret_cast<const f32x4*>(of + (16 * u + m) * RM + 16 * v + 4 * g); };
      const float* vs = reinterpret_cast<const float*>(im + I::kV) + 4 * g * VS + 16 * cw + m;
      auto rest_at = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          scale[u] = token(I::kScale, u);
          pre[u] = token(I::kPrefix, u);
          rest[u] = token(I::kRest, u);
          suffix[u] = token(I::kSuffix, u);
#pragma unroll
          for (int e = 0; e < 4; ++e) w[u][e] = vs[(16 * u + e) * VS];
        }
        a00 = row(A, 0, 0);
        a10 = row(A, 1, 0);
        a11 = row(A, 1, 1);
        if constexpr (DELTA) {
          m00 = row(M, 0, 0);
          t10 = row(M, 1, 0);
          m11 = row(M, 1, 1);
        }
        total = *reinterpret_cast<const float*>(tk + I::kPrefix + 4 * (CW - 1));
      };
      rows_at(0);
      state_at(0);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        __builtin_amdgcn_sched_barrier(0);
        if (kb + 1 < KB) {
          rows_at(kb + 1);
          state_at(kb + 1);
        } else {
          rest_at();
        }
        add_products(rows[kb & 1], sp[kb & 1], sum);
        constexpr int products = NX * (NP == 1 ? 3 : 6), reads = 2 * NX * NP;
#pragma unroll
        for (int i = 0; i < products; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (i < reads || kb + 1 == KB) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          if (kb + 1 < KB) __builtin_amdgcn_sched_group_barrier(0x002, (56 + products - 1) / products, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      lds_barrier();                                      // (the next chunk's rows are there)
      const int n = rows_of(c);
      f32x4 x[2], within[2], across;                      // x (delta rule): what M is multiplied with; across: what the second tile has of the first
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if constexpr (DELTA) {
          f32x4 read = (sum[2 + u][0] + sum[2 + u][1]) * pre[u];
          if (u == 1) {
            f32x4 t = zero;
            across = within[0] = zero;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              t = mma4(t10[e], w[0][e], t);
              across = mma4(a10[e], w[0][e], across);
              within[0] = mma4(a00[e], w[0][e], within[0]);
            }
            read += t;
          }
          x[u] = scale[u] * (w[u] - read);
          w[u] = times_rows(u ? m11 : m00, x[u]);
        } else {
          w[u] *= scale[u];
        }
      }
      if constexpr (!DELTA) {
        across = within[0] = zero;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          across = mma4(a10[e], w[0][e], across);
          within[0] = mma4(a00[e], w[0][e], within[0]);
        }
      }
      within[1] = times_rows(a11, w[1]);
      auto results = [&](const f32x4 (&before)[2], const f32x4 (&low)[2], const f32x4 (&pre)[2], const f32x4 (&rest)[2], const f32x4 (&within)[2], f32x4 across, f32x4 (&result)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float in = within[u][e], more = u ? across[e] : 0.f;
            if constexpr (NP == 3) {                      // (the delta rule)
              const float read = before[u][e] + low[u][e];
              result[u][e] = __builtin_fmaf(read, pre[u][e], __builtin_fmaf(read, rest[u][e], in + more));
            } else {                                      // (in double: the operands' products are exact, and a rounding here shows.  3 % of the time)
              const double p = (double)pre[u][e] + (double)rest[u][e];
              result[u][e] = (float)__builtin_fma((double)before[u][e], p, __builtin_fma((double)low[u][e], p, (double)in + (double)more));
            }
          }
      };
      auto write = [&](const f32x4 (&result)[2]) __attribute__((always_inline)) {
        if (col < a.V) {
          if (n == CW) {                                  // (no question for every row: they took longer than the products)
#pragma unroll
            for (int i = 0; i < 8; ++i) out[4 * i * out_row] = result[i >> 2][i & 3];
          } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
              if (4 * i + g < n) out[4 * i * out_row] = result[i >> 2][i & 3];
          }
        }
      };
      f32x4 result[2];
      results({sum[0][0], sum[1][0]}, {sum[0][1], sum[1][1]}, pre, rest, within, across, result);
      write(result);
      auto parts_of = [&](const f32x4 (&w)[2], const f32x4 (&suffix)[2], u16x8 (&wp)[3]) __attribute__((always_inline)) {
        u16x4 w0[3], w1[3];
        split(w[0] * suffix[0], w0);
        split(w[1] * suffix[1], w1);
#pragma unroll
        for (int p = 0; p < 3; ++p) wp[p] = both(w0[p], w1[p]);
      };
      // Numbers that are not finite: in the state (a row of q times it is none then), in w or in a token's keys (q k of a token with itself, so its row of A w).
      // The chunk is gone through again below, from the state as it is here, which its slot keeps.  (Behind the results: the branch would wait for them.)
      const bool wild = some_not_finite(within[0]) || some_not_finite(within[1]) || (!DELTA && __builtin_amdgcn_ballot_w64(!__builtin_isfinite(sum[0][0][0])));
      if (wild) st.store(slot, a.K, a.V, col, g);
      u16x8 wp[3];
      parts_of(w, suffix, wp);
      // the transposing reads: lane 4 q + p of a group of 16 brings row 4 g + q (and the row 16 below it), keys 16 kt + 4 p ..
      auto keys_of = [&](int kt, u16x8 (&x)[NP]) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          const char* at = im + I::kK + p * I::kPlane + place_of(4 * g + (m >> 2)) * I::kRow + 32 * kt + 8 * (m & 3);
          x[p] = both(lds_tr_read(at), lds_tr_read(at + 16 * I::kRow));
        }
      };
      u16x8 kx[2][4][NP];
      auto keys_at = [&](int k2) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) keys_of(4 * k2 + i, kx[k2 & 1][i]);
      };
      keys_at(0);
#pragma unroll
      for (int k2 = 0; k2 < KT / 4; ++k2) {
        __builtin_amdgcn_sched_barrier(0);
        if (k2 + 1 < KT / 4) keys_at(k2 + 1);
        f32x4 more[4][2] = {{zero, zero}, {zero, zero}, {zero, zero}, {zero, zero}};
        add_products(kx[k2 & 1], wp, more);
        constexpr int products = 4 * (NP == 1 ? 3 : 6);
#pragma unroll
        for (int i = 0; i < products; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (k2 + 1 < KT / 4 && i < 8 * NP) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) st.S[4 * k2 + i][e] = __builtin_fmaf(st.S[4 * k2 + i][e], total, more[i][0][e] + more[i][1][e]);
      }
      if (wild) {                                         // token by token where nothing may reach earlier ones, infinities as what they are
        __builtin_amdgcn_sched_barrier(0);
        st.load(slot, a.K, a.V, col, g, false);
        f32x4 s[NX][2], total_s[NX], w[2], pre[2], rest[2], suffix[2], within[2], across = zero;
#pragma unroll
        for (int i = 0; i < NX; ++i) s[i][0] = s[i][1] = zero;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          __builtin_amdgcn_sched_barrier(0);
          u16x8 x[NX][NP];
#pragma unroll
          for (int i = 0; i < NX; ++i) parts_at(im + (i < 2 ? I::kQ : I::kK), i & 1, kb, x[i]);
          state_at(kb);
          add_products(x, sp[kb & 1], s);
        }
#pragma unroll
        for (int i = 0; i < NX; ++i) total_s[i] = total_of(s[i]);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          pre[u] = token(I::kPrefix, u);
          rest[u] = token(I::kRest, u);
          suffix[u] = token(I::kSuffix, u);
          const f32x4 scale = token(I::kScale, u);
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = vs[(16 * u + e) * VS];
          if constexpr (DELTA) {
            f32x4 read = total_s[2 + u] * pre[u];
            if (u == 1) read += times_rows(row(M, 1, 0), w[0]);
            w[u] = rows_in_order(M + 16 * u * RM + 16 * u, m, g, scale * (v - read), zero);
          } else {
            w[u] = v * scale;
          }
          if (u == 1) across = times_rows(row(A, 1, 0), w[0]);
          within[u] = rows_in_order(A + 16 * u * RM + 16 * u, m, g, w[u], zero);
        }
        f32x4 result[2];
        results({total_s[0], total_s[1]}, {zero, zero}, pre, rest, within, across, result);
        write(result);
        parts_of(w, suffix, wp);
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
          __builtin_amdgcn_sched_barrier(0);
          u16x8 x[1][NP];
          keys_of(kt, x[0]);
#pragma unroll
          for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int e = 0; e < 8; ++e) x[0][p][e] = 4 * e + g < n ? x[0][p][e] : u16(0);      // (rows past the portion: no zeros of theirs meet its last key)
          f32x4 more[1][2] = {{zero, zero}};
          add_products(x, wp, more);
          const f32x4 t = total_of(more[0]);
#pragma unroll
          for (int e = 0; e < 4; ++e) st.S[kt][e] = __builtin_fmaf(st.S[kt][e], total, t[e]);
        }
      }
      out += CW * out_row;
    }
    st.store(slot, a.K, a.V, col, g);
    return;
  }

  // Producers
  const int tid = (int)threadIdx.x, qk_head = head / (a.heads / a.qk_heads);
  const typename QK::storage* q = (const typename QK::storage*)a.q + t_begin * a.q_stride + (int64_t)qk_head * a.K;
  const typename QK::storage* k = (const typename QK::storage*)a.k + t_begin * a.k_stride + (int64_t)qk_head * a.K;
  const typename VT::storage* v = (const typename VT::storage*)a.v + t_begin * a.v_stride + (int64_t)head * a.V;
  const bool scaled = DELTA || a.vscale;
  const float* per_token = DELTA ? a.beta : a.vscale ? a.vscale : a.decay;
  constexpr int NQ = CW * KP / 4 / 256, NV = CW * VW / 4 / 256;
  auto qk_row = [&](int i) { return (tid + 256 * i) / (KP / 4); };
  auto qk_col = [&](int i) { return (tid + 256 * i) % (KP / 4) * 4; };
  auto v_row = [&](int i) { return (tid + 256 * i) / (VW / 4); };
  const int v_col = tid % (VW / 4) * 4;
  struct Set {
    Piece<QK, 4, VEC> q[NQ], k[NQ];
    Piece<VT, 4, VEC> v[NV];
    float scale;
  } next;                                                 // the chunk's whose rows are on their way
  // (strides below 2^28: what chunk_scan.hip sends here)
  auto at_row = [&](auto* base, int r, int64_t stride) __attribute__((always_inline)) {
    typedef std::remove_pointer_t<decltype(base)> E;
    return reinterpret_cast<E*>(reinterpret_cast<const char*>(base) + (uint64_t)(uint32_t)r * (uint32_t)(stride * sizeof(E)));
  };
  auto fetch = [&](Set& s, int chunk) __attribute__((always_inline)) {
    if (chunk >= n_chunks) return;                        // (what is there stays, and nobody looks at it)
    const int n = rows_of(chunk);                         // rows past the portion repeat its last one
    const int64_t t0 = (int64_t)chunk * CW;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      s.q[i].load(at_row(q + t0 * a.q_stride, min(qk_row(i), n - 1), a.q_stride), qk_col(i), a.K);
      s.k[i].load(at_row(k + t0 * a.k_stride, min(qk_row(i), n - 1), a.k_stride), qk_col(i), a.K);
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) s.v[i].load(at_row(v + t0 * a.v_stride, min(v_row(i), n - 1), a.v_stride), col0 + v_col, a.V);
    s.scale = per_token[(t_begin + t0 + min(tid & (CW - 1), n - 1)) * a.heads + head];
  };
  auto decay_at = [&](int chunk) __attribute__((always_inline)) {      // of token lane % 32
    const int n = chunk < n_chunks ? rows_of(chunk) : 1, t = lane & (CW - 1);
    const float d = a.decay[(t_begin + (int64_t)min(chunk, n_chunks - 1) * CW + min(t, n - 1)) * a.heads + head];
    return t < n ? d : 1.f;
  };
  // (rows past the portion repeat its last one: the values and write strengths there are none)
  const bool whole = a.K == KP;
  auto planes = [&](char* to, const Piece<QK, 4, VEC>& p, int at) __attribute__((always_inline)) {
    const int col = qk_col(at);
    f32x4 x;
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = QK::to_float(p.r[j]);
    if (!whole) {
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = col + j < a.K ? x[j] : 0.f;
    }
    char* dst = to + place_of(row_of(qk_row(at))) * I::kRow + 2 * col;
    if constexpr (NP == 1) {
      *reinterpret_cast<u16x4*>(dst) = u16x4{BF16::from_float(x[0]), BF16::from_float(x[1]), BF16::from_float(x[2]), BF16::from_float(x[3])};
    } else {
      u16x4 part[3];
      split(x, part);
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<u16x4*>(dst + i * I::kPlane) = part[i];
    }
  };
  auto store = [&](const Set& s, int chunk) __attribute__((always_inline)) {
    const int n = rows_of(chunk);
    char* im = image(chunk);
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      planes(im + I::kQ, s.q[i], i);
      planes(im + I::kK, s.k[i], i);
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      f32x4 f;
#pragma unroll
      for (int j = 0; j < 4; ++j) f[j] = s.v[i].get(j, v_row(i) < n, col0 + v_col, a.V);
      *reinterpret_cast<f32x4*>(im + I::kV + 4 * (row_of(v_row(i)) * VS + v_col)) = f;
    }
    if (tid < CW) reinterpret_cast<float*>(tokens(chunk) + I::kScale)[row_of(tid)] = tid >= n ? (DELTA ? 0.f : 1.f) : scaled ? s.scale : 1.f;      // (a row past the portion changes nothing)
  };
  const int t_m = row_of_token(m);
  // (x k^T)[i, j] of two tiles with rows i = 4 g + e and column j = m: tokens 4 e + g and t_m of theirs.  N products that share one operand, the keys
  // (SECOND: the rows); `of` and `with`: offsets of planes and tiles.
  struct Tile { int planes, u; };
  auto block_products = [&](const char* im, const auto& of, Tile with, auto second, auto& xk) __attribute__((always_inline)) {
    constexpr int N = std::extent_v<std::remove_reference_t<decltype(xk)>>;
    f32x4 sum[N][2];
#pragma unroll
    for (int i = 0; i < N; ++i) sum[i][0] = sum[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    u16x8 x[2][N][NP], y[2][NP];
    auto read = [&](int kb) __attribute__((always_inline)) {
      parts_at(im + with.planes, with.u, kb, y[kb & 1]);
#pragma unroll
      for (int i = 0; i < N; ++i) parts_at(im + of[i].planes, of[i].u, kb, x[kb & 1][i]);
    };
    read(0);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      __builtin_amdgcn_sched_barrier(0);
      if (kb + 1 < KB) read(kb + 1);
      add_products<decltype(second)::value>(x[kb & 1], y[kb & 1], sum);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) xk[i] = sum[i][0] + sum[i][1];
  };
  // Products of a tile's decays behind token `from` and up to the lane's four rows; and to the tile's end
  struct Runs { Product mine[4], behind; };
  auto runs = [&](const float (&d)[C], int from) __attribute__((always_inline)) {
    Runs r;
#pragma unroll
    for (int t = 0; t < C; ++t) {
      r.behind.by(t > from ? d[t] : 1.f);
      const bool here = (t & 3) == 0 || (t & 3) == g;
      r.mine[t >> 2].hi = here ? r.behind.hi : r.mine[t >> 2].hi;
      r.mine[t >> 2].lo = here ? r.behind.lo : r.mine[t >> 2].lo;
    }
    return r;
  };
  auto decays = [&](float decay, int u, float (&d)[C]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < C; ++t) d[t] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, decay), 16 * u + t));
  };
  // What depends on the decays alone, while the consumers have products to make; each product of decays is rounded once.  Wave 0: A_00, T_10, prefixes
  // and the first tile's suffixes; wave 1: A_11, A_10 and the second's; waves 2 and 3: M_00 and M_11.
  struct Factors {
    Product own[4], across[4];      // (waves 2 and 3: own[.].hi alone)
  } f;
  auto make_factors = [&](float decay, char* tk) __attribute__((always_inline)) {
    float d0[C], d1[C];
    if (wave == 0) {
      decays(decay, 0, d0);
      decays(decay, 1, d1);
      const Runs first = runs(d0, t_m), second = runs(d1, -1);
      Product up_to = first.behind;                       // (t_m = 0: all of the first tile's)
      up_to.by(d0[0]);
      f32x4 prefix[2], rest[2];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f.own[e] = first.mine[e];
        f.across[e] = product_of(second.mine[e], first.behind);
        Product p[2] = {first.mine[e], product_of(second.mine[e], up_to)};
        p[0].by(d0[0]);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          prefix[u][e] = p[u].value();
          rest[u][e] = (p[u].hi - prefix[u][e]) + p[u].lo;
        }
      }
      if (m == 0) {                                       // (t_m = 0)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          *reinterpret_cast<f32x4*>(tk + I::kPrefix + 4 * (16 * u + 4 * g)) = prefix[u];
          *reinterpret_cast<f32x4*>(tk + I::kRest + 4 * (16 * u + 4 * g)) = rest[u];
        }
      }
      if (g == 0) reinterpret_cast<float*>(tk + I::kSuffix)[m] = product_of(first.behind, second.behind).value();
    } else if (wave == 1) {
      decays(decay, 0, d0);
      decays(decay, 1, d1);
      const Product behind = runs(d0, t_m).behind;
      const Runs own = runs(d1, t_m), second = runs(d1, -1);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f.own[e] = own.mine[e];
        f.across[e] = product_of(second.mine[e], behind);
      }
      if (g == 0) reinterpret_cast<float*>(tk + I::kSuffix)[16 + m] = own.behind.value();
    } else if constexpr (DELTA) {
      decays(decay, wave - 2, d0);
      float run = 1.f;
#pragma unroll
      for (int t = 0; t < C; ++t) {
        run = t > t_m ? run * d0[t] : 1.f;
        f.own[t >> 2].hi = (t & 3) == 0 || (t & 3) == g ? run : f.own[t >> 2].hi;
      }
    }
  };
  auto make_M = [&](char* im, const char* tk, int u, f32x4 kk) __attribute__((always_inline)) {
    float* M = reinterpret_cast<float*>(im + I::kM) + 16 * u * RM + 16 * u;      // T (by tokens), then M
    const f32x4 b = *reinterpret_cast<const f32x4*>(tk + I::kScale + 4 * (16 * u + 4 * g));
#pragma unroll
    for (int e = 0; e < 4; ++e) M[(4 * e + g) * RM + t_m] = t_m < 4 * e + g ? b[e] * kk[e] * f.own[e].hi : 0.f;
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
        const f32x4 T = *reinterpret_cast<const f32x4*>(M + t * RM + s);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (s + e >= t) continue;
          if (e & 1) s1 -= T[e] * x[s + e];
          else s0 -= T[e] * x[s + e];
        }
      }
      x[t] = s0 + s1;
      if (t == 5 || t == 8 || t == 11 || t == 13) asm volatile("" ::: "memory");      // (a few rows of T in registers at a time, not all of them)
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();                      // T has been read
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (g == 0) {
#pragma unroll
      for (int t = 0; t < C; ++t) M[row_of_token(t) * RM + m] = x[t];
    }
  };
  fetch(next, 0);
  float decay = decay_at(0);
  for (int c = 0; c < n_chunks; ++c) {
    make_factors(decay, tokens(c));
    store(next, c);
    if (!DELTA) fetch(next, c + 1);
    decay = decay_at(c + 1);
    lds_barrier();
    char* im = image(c);
    f32x4 xk[2];
    if (wave == 0) {
      if constexpr (DELTA) {
        const Tile of[2] = {{I::kQ, 0}, {I::kK, 1}};
        block_products(im, of, Tile{I::kK, 0}, std::false_type(), xk);
      } else {
        f32x4 qk[1];
        const Tile of[1] = {{I::kQ, 0}};
        block_products(im, of, Tile{I::kK, 0}, std::false_type(), qk);
        xk[0] = qk[0];
      }
    } else if (wave == 1) {
      const Tile of[2] = {{I::kK, 1}, {I::kK, 0}};
      block_products(im, of, Tile{I::kQ, 1}, std::true_type(), xk);
    } else if constexpr (DELTA) {
      f32x4 kk[1];
      const Tile of[1] = {{I::kK, wave - 2}};
      block_products(im, of, of[0], std::false_type(), kk);
      xk[0] = kk[0];
    }
    if (DELTA) fetch(next, c + 1);                        // (behind the products, which want the registers)
    float *A = reinterpret_cast<float*>(im + I::kA) + 4 * g * RM + m, *M = reinterpret_cast<float*>(im + I::kM) + 4 * g * RM + m;
    if (wave < 2) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        A[(16 * wave + e) * RM + 16 * wave] = t_m <= 4 * e + g ? f.own[e].times(xk[0][e]) : 0.f;
        if (wave == 1) A[(16 + e) * RM] = f.across[e].times(xk[1][e]);
        else if constexpr (DELTA) M[(16 + e) * RM] = f.across[e].times(xk[1][e]);
      }
    } else if constexpr (DELTA) {
      make_M(im, tokens(c), wave - 2, xk[0]);
    }
    lds_barrier();
  }
  lds_barrier();                                          // (the consumers' last)
}

template <int KP, bool DELTA, typename QK, typename VT, bool VEC>
int launch(const ChunkScanArgs& a, hipStream_t s) {
  return launch_chunks(chunk_head32_kernel<KP, DELTA, QK, VT, VEC>, dim3((unsigned)a.heads, (unsigned)((a.V + VW - 1) / VW), (unsigned)a.n_seq), 512,
                       HeadImage<KP, QK, DELTA>::kLds, a, s);
}
// (what chunk_scan.hip sends here: the delta rule with more than 64 key channels, and the decayed sum of bfloat16 q and k)
template <int KP, typename QK, typename VT, bool VEC>
int launch_form(const ChunkScanArgs& a, hipStream_t s) {
  if (a.form == hxm::kChunkDelta) {
    if constexpr (KP == 128) return launch<KP, true, QK, VT, VEC>(a, s);
  } else {
    if constexpr (QK::kDtype == HX_BF16) return launch<KP, false, QK, VT, VEC>(a, s);
  }
  return HX_ERR_UNSUPPORTED;
}
template <typename QK, typename VT>
int launch_width(const ChunkScanArgs& a, hipStream_t s) {
  const bool vec = rows_by_four(a);
  if (a.K <= 64) return vec ? launch_form<64, QK, VT, true>(a, s) : launch_form<64, QK, VT, false>(a, s);
  return vec ? launch_form<128, QK, VT, true>(a, s) : launch_form<128, QK, VT, false>(a, s);
}

}  // namespace

namespace hxm {

int chunk_head(const ChunkScanArgs& a, hipStream_t s) {
  if (a.q_dtype == HX_BF16) return launch_width<BF16, BF16>(a, s);
  return a.v_dtype == HX_F32 ? launch_width<F32, F32>(a, s) : launch_width<F32, BF16>(a, s);
}

}  // namespace hxm
