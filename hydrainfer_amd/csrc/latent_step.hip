// latent_step.hip — latent attention of batches of single tokens (bfloat16, latents of 64 KK columns, up to 32 heads, pages of whole
// 16-row groups): a workgroup takes a run of one token's keys, all of its heads over it.  The form of row tiles (latent_attn.hip) gives
// a wave 16 rows of token and head for all of a tile's keys: with 8 to 32 rows a token two or three of its four waves stand idle, the others go
// through keys, softmax and values alone, and what they wait for in front of the first product are five loads behind each other.
// Here a tile is 64 keys, in the scores wave w takes 16 of them (for 16 heads), in the values a quarter of the columns; scores
// pass between the two through LDS as floats, so that every wave makes the weights it needs itself and a tile costs two barriers, and one more where another tile comes into its place.
// A weight enters the second product as the sum of two bfloat16 numbers (p = hi + lo, relative 2^-17): it costs matrix time that is idle here and the
// results' own rounding is all that is left.
// Latency bounds it: the way to the first tile, then for each tile keys, softmax and values in turn, and the launch that merges.  Measured, 32 tokens
// of 301 - 1747 keys under a window of 512, 512 columns, 32 heads: 21.1 us in the row tiles' form, 15.6 here, 3 to 5 of it the merge (17.7 with every
// wave fetching its queries itself); without the window 28.7 and 23.9; 1 token behind 149 keys 14.9 and 9.6; 51 tokens of 26 - 87 keys, 64
// columns, 8 heads 6.2 and 4.5.
// Tiles go straight from the paged cache to LDS, N_BUF of them at a time, as chunks of 16 bytes in the places that the wide form's rows have.
#include <algorithm>

#include "attn_common.h"
#include "latent_step.h"

namespace hxm {
int& last_hip_error();
int check_launch();
}

namespace {

using namespace hx;

constexpr int kTile = 64;                  // keys of a tile
constexpr int kScoreRow = kTile + 4;       // floats of a head's scores in LDS: rows of 16 bytes that start in different banks
constexpr float kLog2e = 1.4426950408889634f;

// Tiles in LDS: one being read, the others on their way.  160 KiB a compute unit; up to 256 columns two workgroups share it.
constexpr int buffers(int KK) { return KK <= 2 ? 4 : KK == 5 || KK == 6 ? 3 : 2; }
constexpr size_t lds_bytes(int KK, int RT) { return (size_t)buffers(KK) * kTile * 128 * KK + (size_t)RT * 16 * kScoreRow * 4; }

template <int KK, int RT>                  // columns / 64, groups of 16 heads
__global__ __launch_bounds__(256 * RT, KK <= 4 ? 2 * RT : RT) void latent_step_kernel(hxm_latent_attn_args a) {
  constexpr int R = 64 * KK, RS = 2 * R, L = R / 8, IMG = kTile * RS, NB = buffers(KK), NW = 4 * RT, KPW = kTile / NW;
  constexpr int KS = R / 32, NDB = R / 64;   // steps of the scores' contraction; blocks of 16 columns a wave has in the values
  constexpr int NL = KPW * L / 64;           // 16-byte chunks a lane asks for, a tile
  constexpr bool FULL = RS % 256 == 0;       // (the places of a row's chunks: latent_attn.hip)
  extern __shared__ __attribute__((aligned(256))) char smem_w[];
  auto swz = [](int row) {
    if (FULL) return (row & 15) < 8 ? 2 * (row & 7) : 31 - 2 * (row & 15);
    const int h = (row & 15) >> 1;
    return h < 4 ? 2 * h : 15 - 2 * h;
  };
  typedef __attribute__((address_space(4))) const int32_t c_i32;       // (uniform indices: through the scalar cache)
  const int t = blockIdx.x, split = blockIdx.y, n_splits = gridDim.y;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = lane & 15, g = lane >> 4, part = wave & 3, rt = wave >> 2;
  const int head = min(16 * rt + c, a.n_heads - 1);      // (rows past the last head repeat it and are not written)
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem_w;
  // The queries come by way of LDS, into the place of tile NB - 1 (each of the four waves that want a row would fetch it in pieces of 64 bytes).
  {
    const char* qg = (const char*)a.q + 2 * (int64_t)t * a.q_token_stride;
    for (int j = wave; j < RT * L / 4; j += NW) {
      const int i = 64 * j + lane, row = i / L, ch = i - row * L;
      const char* from = qg + 2 * (int64_t)min(row, a.n_heads - 1) * a.q_head_stride + 16 * (ch ^ swz(row));
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(__builtin_amdgcn_readfirstlane(lds0 + (uint32_t)((NB - 1) * IMG + 1024 * j))) : "memory", "m0");
#pragma clang diagnostic pop
    }
  }
  // The token's sequence is nearly always the token's own number: its pages are looked up along with it.
  c_i32* cu_blocks = (c_i32*)a.cu_block_lens;
  const int b = ((c_i32*)a.tok_seq)[t], pos = ((c_i32*)a.positions)[t];
  int first_page = cu_blocks[min(t, a.n_seq)];
  if (b != t) first_page = cu_blocks[b];
  const int k_first = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  // this split's run of groups of 16 keys (the last splits may get none)
  const int g_first = k_first >> 4, per = ((pos >> 4) - g_first + n_splits) / n_splits;
  const int key_at = 16 * (g_first + split * per), key_end = pos < 0 ? key_at : min(pos + 1, key_at + 16 * per);
  const int n_tiles = max(0, key_end - key_at + kTile - 1) / kTile;

  const u16* cache = (const u16*)a.cache;
  c_i32* table = (c_i32*)(a.block_table + first_page);
  const int bs = a.block_size, bshift = (bs & (bs - 1)) == 0 ? __ffs(bs) - 1 : -1;
  const uint32_t row_bytes = (uint32_t)(2 * a.cache_row_stride);
  // Wave w brings keys KPW w .. of a tile (one page): rows in front of the first key or behind the last repeat those.
  auto bring = [&](int tile, int img) __attribute__((always_inline)) {
    const int key0 = min(max(key_at + tile * kTile + KPW * wave, k_first & ~(KPW - 1)), (key_end - 1) & ~(KPW - 1));
    const int r_min = k_first - key0, r_max = key_end - 1 - key0;
    const int page = bshift >= 0 ? key0 >> bshift : key0 / bs;
    const u16* base = cache + (int64_t)table[page] * a.cache_block_stride + (int64_t)(key0 - page * bs) * a.cache_row_stride;
    const uint32_t to = lds0 + (uint32_t)(img * IMG + KPW * wave * RS);
    uint32_t ln = (uint32_t)lane;
    asm volatile("" : "+v"(ln));             // (worked out anew every time: kept, the addresses would take the registers of the queries)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    // (m0, the LDS address of the transfer, is a reserved register: nothing else in this kernel uses it)
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      uint32_t off;
      if constexpr (L == 64) {               // a row a load: nothing of it differs from lane to lane but the column
        off = (16u * ln ^ 16u * (uint32_t)swz(KPW * wave + j)) + (uint32_t)max(min(j, r_max), r_min) * row_bytes;
      } else {
        const uint32_t rr = (64u * j + ln) / L, ch = 64u * j + ln - rr * L;
        off = (uint32_t)max(min((int)rr, r_max), r_min) * row_bytes + 16u * (ch ^ (uint32_t)swz(KPW * wave + (int)rr));
      }
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(__builtin_amdgcn_readfirstlane(to + 1024u * j)) : "memory", "m0");
    }
#pragma clang diagnostic pop
  };
#pragma unroll
  for (int i = 0; i < NB - 1; ++i)
    if (i < n_tiles) bring(i, i);
  constexpr int NP = FULL ? 4 : 2;
  // Reads of rows: chunk 4 ks + g of row r; the places of a row's chunks differ in the low four (three) bits of their numbers.
  typedef __attribute__((address_space(3))) const u16x8 lds_row;
  auto row_read = [](uint32_t row0, int ks) __attribute__((always_inline)) {
    return *(lds_row*)(uintptr_t)((row0 ^ (64u * (ks % NP))) + 64u * NP * (ks / NP));
  };
  // (in order: the queries are there when at most the tiles behind them are on their way)
  if (n_tiles >= NB - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - 1) * NL) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  u16x8 qf[KS];                              // the queries (B operand): head c, columns 32 ks + 8 g ..
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qf[ks] = row_read(lds0 + (uint32_t)((NB - 1) * IMG + (16 * rt + c) * RS + 16 * (g ^ swz(c))), ks);
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[ks]));
  __syncthreads();
  if (NB - 1 < n_tiles) bring(NB - 1, NB - 1);
  float scale2 = a.scale * kLog2e;
  if (scale2 < 0.f) {                        // (a maximum of scores is one of scaled scores where the scale is positive)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] ^= (u16)0x8000;
  }
  scale2 = fabsf(scale2) < 1e-30f ? 1e-30f : fabsf(scale2);      // (not fmaxf: what is not a number stays so)
  f32x4 acc[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = HX_NEG_BIG, l = 0.f;
  // Transposing reads: lane 4 q + p of a group of 16 brings row 4 g + q (and the row 16 below it: the same place), columns 16 db + 4 p .. of the wave's quarter.
  const uint32_t kp0 = lds0 + (uint32_t)((16 * part + c) * RS + 16 * (g ^ swz(c)));
  const int vrow = 4 * g + (c >> 2);
  const uint32_t v_at = lds0 + (uint32_t)(vrow * RS + 8 * (c & 1)), v_swz = (uint32_t)swz(vrow), v_ch = (uint32_t)(part * 2 * NDB + ((c & 3) >> 1));
  const uint32_t s0 = lds0 + (uint32_t)(NB * IMG + (16 * rt + c) * kScoreRow * 4);      // this head's scores
  typedef __attribute__((address_space(3))) f32x4 lds_f4;
  typedef __attribute__((address_space(3))) hx_s16x4_t lds_s4;
  auto tr_read = [](uint32_t at) __attribute__((always_inline)) {
    return __builtin_bit_cast(u16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(uintptr_t)at));
  };
  int img = 0;
  for (int tile = 0; tile < n_tiles; ++tile) {
    // this tile is there; the ones behind it, at most NB - 1, may be on their way
    if constexpr (NB == 4) {
      if (tile + 3 < n_tiles) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * NL) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else if constexpr (NB == 3) {
      if (tile + 2 < n_tiles) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NL) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else {
      if (tile + 1 < n_tiles) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NL) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();
    {
      const uint32_t kp = kp0 + (uint32_t)(img * IMG);
      f32x4 s[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) s[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      constexpr int kAhead = KS < 8 ? KS : 8;
      u16x8 kf[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead; ++i) kf[i] = row_read(kp, i);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        s[i & 1] = Mfma<BF16>::mma(kf[i % kAhead], qf[i], s[i & 1]);
        if (i + kAhead < KS) kf[i % kAhead] = row_read(kp, i + kAhead);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) s[0][e] += s[1][e];
      *(lds_f4*)(uintptr_t)(s0 + (uint32_t)(16 * part + 4 * g) * 4) = s[0];      // keys 16 part + 4 g .. of head c
    }
    __syncthreads();
    const int key_l = key_at + tile * kTile + 4 * g;       // element e of group u: key key_l + 16 u + e
    f32x4 p[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) p[u] = *(lds_f4*)(uintptr_t)(s0 + (uint32_t)(16 * u + 4 * g) * 4);
    const int last = key_end - 1 - key_l, first = k_first - key_l;
    float mx = HX_NEG_BIG;
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (16 * u + e > last || 16 * u + e < first) p[u][e] = -INFINITY;
        mx = fmaxf(mx, p[u][e]);
      }
    mx = groups_max(mx);
    float m_ref = mx * scale2;
    asm("" : "+v"(m_ref));                   // (rounded: left inside a difference below it would not be the maximum's number)
    const float m_new = fmaxf(m, m_ref), alpha = fast_exp2(m - m_new);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int i = 0; i < NDB; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][e] *= alpha;
    u16x8 hi[2], lo[2];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float w = fast_exp2(__builtin_fmaf(p[u][e], scale2, -m));
        l += w;
        const u16 h = BF16::from_float(w);
        hi[u >> 1][4 * (u & 1) + e] = h;
        lo[u >> 1][4 * (u & 1) + e] = BF16::from_float(w - BF16::to_float(h));
      }
    const uint32_t va = v_at + (uint32_t)(img * IMG);
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {       // rows 32 ks + 4 g + q, and those 16 below
        const uint32_t at = va + 16u * ((v_ch + 2 * db) ^ v_swz) + (uint32_t)(32 * ks) * RS;
        const u16x4 x0 = tr_read(at), x1 = tr_read(at + 16u * RS);
        const u16x8 x = u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
        acc[db] = Mfma<BF16>::mma(x, hi[ks], acc[db]);
        acc[db] = Mfma<BF16>::mma(x, lo[ks], acc[db]);
      }
    if (tile + NB < n_tiles) {
      __syncthreads();                       // everybody has read this tile
      bring(tile + NB, img);
    }
    img = img + 1 == NB ? 0 : img + 1;
  }
  float total = l + __shfl_xor(l, 16, 64);
  total += __shfl_xor(total, 32, 64);
  if (16 * rt + c >= a.n_heads) return;
  const int col0 = part * (R / 4) + 4 * g;   // O[head c][column col0 + 16 db + e]
  if (n_splits > 1) {                        // what this split adds, not normalised: ws_o [token][16 RT rows][split][R], ws_ml [..][split][maximum (log2), sum]
    const size_t at = ((size_t)t * (16 * RT) + head) * n_splits + split;
    float* wo = a.ws_o + at * R + col0;
#pragma unroll
    for (int db = 0; db < NDB; ++db) *reinterpret_cast<f32x4*>(wo + 16 * db) = acc[db];
    if (part == 0 && g == 0) {
      a.ws_ml[2 * at] = m;
      a.ws_ml[2 * at + 1] = total;
    }
    return;
  }
  if (a.sinks) total += fast_exp2(a.sinks[head] * kLog2e - m);      // the sink: one more term, without a value
  float gsc = 1.0f / total;
  if (a.gate_pre) gsc = gsc / (1.0f + __expf(-BF16::to_float(((const u16*)a.gate_pre)[(int64_t)t * a.gate_stride + head])));
  u16* og = (u16*)a.out + (int64_t)t * a.out_token_stride + (int64_t)head * a.out_head_stride + col0;
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
    u16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = BF16::from_float(acc[db][e] * gsc);
    *reinterpret_cast<u16x4*>(og + 16 * db) = o;
  }
}

// The splits of a row merged: out = sum_s O_s 2^(m_s - M) / sum_s l_s 2^(m_s - M), times the head gate.  A row to `lanes` lanes of four
// columns; every load of a pass of eight splits is in flight at once.
__global__ __launch_bounds__(256) void latent_step_merge_kernel(hxm_latent_attn_args a, int rows, int n_splits, int lanes_log2) {
  const int R = a.kv_rank, lanes = 1 << lanes_log2;
  const uint32_t item = blockIdx.x * (256u >> lanes_log2) + (threadIdx.x >> lanes_log2);
  const int t = (int)(item / (uint32_t)a.n_heads), h = (int)(item % (uint32_t)a.n_heads);
  if (t >= a.n_tokens) return;
  const size_t row = (size_t)t * rows + h;
  const float* ml = a.ws_ml + 2 * row * n_splits;
  float gate = 1.f;
  if (a.gate_pre) gate = 1.0f / (1.0f + __expf(-BF16::to_float(((const u16*)a.gate_pre)[(int64_t)t * a.gate_stride + h])));
  u16* og = (u16*)a.out + (int64_t)t * a.out_token_stride + (int64_t)h * a.out_head_stride;
  for (int c = 4 * ((int)threadIdx.x & (lanes - 1)); c < R; c += 4 * lanes) {
    const float* wo = a.ws_o + row * n_splits * R + c;
    f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
    float M = HX_NEG_BIG, total = 0.f;
    for (int s0 = 0; s0 < n_splits; s0 += 8) {
      float mx[8], l[8];
      f32x4 v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int s = min(s0 + i, n_splits - 1);
        v[i] = *reinterpret_cast<const f32x4*>(wo + (size_t)s * R);
        mx[i] = ml[2 * s];
        l[i] = ml[2 * s + 1];
      }
      float m_new = M;
#pragma unroll
      for (int i = 0; i < 8; ++i) m_new = fmaxf(m_new, mx[i]);
      const float keep = fast_exp2(M - m_new);
      total *= keep;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] *= keep;
      M = m_new;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float w = s0 + i < n_splits ? fast_exp2(mx[i] - M) : 0.f;
        total += w * l[i];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] += w * v[i][e];
      }
    }
    if (a.sinks) total += fast_exp2(a.sinks[h] * kLog2e - M);      // the sink counts once, here
    const float gsc = gate / total;
    *reinterpret_cast<u16x4*>(og + c) = u16x4{BF16::from_float(o[0] * gsc), BF16::from_float(o[1] * gsc), BF16::from_float(o[2] * gsc), BF16::from_float(o[3] * gsc)};
  }
}

template <int KK, int RT>
int launch(const hxm_latent_attn_args& a, hipStream_t s) {
  constexpr size_t lds = lds_bytes(KK, RT);
  const int n_splits = a.n_splits > 1 ? a.n_splits : 1;
  auto kernel = latent_step_kernel<KK, RT>;
  if (lds > 48 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
      hxm::last_hip_error() = (int)e;
      return HX_ERR_HIP;
    }
  }
  kernel<<<dim3((unsigned)a.n_tokens, (unsigned)n_splits), dim3(256 * RT), lds, s>>>(a);
  if (n_splits > 1) {
    int lanes_log2 = 4;                      // a row to R / 4 lanes, at most a power of two of them
    while ((8 << lanes_log2) <= a.kv_rank && lanes_log2 < 7) ++lanes_log2;
    const int64_t threads = ((int64_t)a.n_tokens * a.n_heads) << lanes_log2;
    latent_step_merge_kernel<<<dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s>>>(a, 16 * RT, n_splits, lanes_log2);
  }
  return hxm::check_launch();
}

template <int KK>
int launch_heads(const hxm_latent_attn_args& a, hipStream_t s) {
  return a.n_heads <= 16 ? launch<KK, 1>(a, s) : launch<KK, 2>(a, s);
}

}  // namespace

namespace hxm {

// Up to 2048 tiles of keys in all, 1365 for more than 16 heads and 64 tokens: behind that the compute units are full, and what counts is not the way to
// the first tile but how many rows a byte from LDS feeds, which are more in the row tiles' form (us there and here, 32 heads: 192 tokens of 200 - 2047 keys, 128
// columns 29.6 43.2, 320 columns 53 69; 512 under a window of 512, 320 columns 47 56; 64 of 1000 - 8000, 128 columns 37 46; in front of the line, 512 columns, 128 of
// 26 - 300 27.7 19.7, 64 of 200 - 2047 41 35).  Of 2337 batches of 1 - 768 tokens behind 17 - 16000 keys 1370 lie in front of it: 0.78 of that form's time in the mean, 8 of them
// 2 - 9 % more.
bool latent_step_serves(const hxm_latent_attn_args& a) {
  if (a.max_q_len != 1 || a.n_tokens > a.n_seq || a.n_heads > 32) return false;
  const int reach = a.window > 0 && a.window < a.max_kv_len ? a.window + 1 : a.max_kv_len;
  return (int64_t)a.n_tokens * ((std::max(reach, 1) + kTile - 1) / kTile) <= (a.n_heads <= 16 || a.n_tokens <= 64 ? 2048 : 1365);
}

// Splits of a token's keys: a launch lasts as long as its rounds of workgroups (256 of more than 256 columns at a time, 512 of fewer), a round
// about 6 us and its tiles, the merge 3 us and what the splits hold.  Only splits of whole tiles are looked at: half a tile costs a whole one.
// The constants (nanoseconds) are fitted to 120 shapes of 1 - 64 tokens behind 26 - 2047 keys, 8, 16 and 32 heads, 64 - 512 columns, each at 17
// splits: 1 % above the best of them in the mean, 9 % at most, and 0.74 of the row tiles' form's times (64 tokens of 200 - 2047 keys, 8 heads, 320 columns:
// 1.01; everything else is faster).
int latent_step_splits(const hxm_latent_attn_args& a) {
  const int reach = a.window > 0 && a.window < a.max_kv_len ? a.window + 1 : a.max_kv_len;
  if (reach <= kTile || a.n_tokens < 1) return 1;
  // (a window's first key may lie anywhere in its group of 16)
  const uint32_t groups = (uint32_t)(reach + 15) / 16 + (reach < a.max_kv_len ? 1 : 0), slots = a.kv_rank > 256 ? 256 : 512;
  const int64_t R = a.kv_rank, head_groups = a.n_heads <= 16 ? 1 : 2;
  const int64_t fixed = 6000 + 1300 * R * head_groups / 512, tile = 650 + 500 * R / 512 + 900 * R * head_groups / 512;
  const int64_t merged = (int64_t)a.n_tokens * a.n_heads * R * 6000 / (160 * 32 * 512);
  int64_t best = 0;
  int splits = 1;
  for (uint32_t ns = std::min((groups + 3) / 4, 64u); ns >= 1; --ns) {
    const uint32_t tiles = (groups + 4 * ns - 1) / (4 * ns);
    if (ns > 1 && (ns - 1) * tiles * 4 >= groups) continue;      // (fewer splits do with as many tiles each)
    const int64_t rounds = ((uint32_t)a.n_tokens * ns + slots - 1) / slots;
    const int64_t cost = rounds * (fixed + tiles * tile) + (ns > 1 ? 2800 + (110 + merged) * ns : 0);
    if (!best || cost < best) {
      best = cost;
      splits = (int)ns;
    }
  }
  return splits;
}

int launch_latent_step(const hxm_latent_attn_args& a, hipStream_t s) {
  if (a.n_splits > 1 && (a.n_splits > 64 || !a.ws_o || !a.ws_ml)) return HX_ERR_WORKSPACE;
  switch (a.kv_rank / 64) {
    case 1: return launch_heads<1>(a, s);
    case 2: return launch_heads<2>(a, s);
    case 3: return launch_heads<3>(a, s);
    case 4: return launch_heads<4>(a, s);
    case 5: return launch_heads<5>(a, s);
    case 6: return launch_heads<6>(a, s);
    case 7: return launch_heads<7>(a, s);
    default: return launch_heads<8>(a, s);
  }
}

}  // namespace hxm
