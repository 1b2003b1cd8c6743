// latent_attn.hip — attention over a paged cache of low-rank latents.  A token leaves ONE row c (kv_rank numbers) in the
// cache; every head's key and value are linear maps of it, so with the key map folded into the query (q~ = W_uk^T q) and
// the value map applied afterwards (o = W_uv sum_j p_j c_j) the kernel is multi-query attention whose keys and values
// are the same rows: score = q~ . c_j * scale, out = sum_j softmax(score)_j c_j.  Scores, weights and sums are float.
// Sliding window: a query at position i sees keys j with 0 <= i - j < window.
#include "attn_common.h"
#include "latent_step.h"
#include "../../include/hydra_mix.h"

namespace hxm {
int& last_hip_error();
int check_launch();
int& tile_form();      // 0: row form only (A/B measurements), 1: tile form where it applies
}

namespace {

using namespace hx;

// one WAVE per token (four tokens a workgroup, no barriers): both latents of the token from its projection row.  vec:
// every pointer, offset and stride lets a lane move four elements at a time.
template <typename A>
__global__ __launch_bounds__(256) void latent_norm_cache_kernel(const typename A::storage* __restrict__ proj, int64_t proj_stride,
                                                                int64_t q_off, int64_t q_rank, int64_t kv_off, int64_t kv_rank,
                                                                const float* __restrict__ q_w, const float* __restrict__ kv_w, float eps,
                                                                typename A::storage* __restrict__ cq_out,
                                                                const int32_t* __restrict__ slot_ids,
                                                                typename A::storage* __restrict__ cache, int64_t cache_block_stride,
                                                                int64_t cache_row_stride, int32_t block_size, int64_t n_tokens, int vec) {
  typedef typename A::storage ST;
  typedef ST ST4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= n_tokens) return;
  const ST* p = proj + t * proj_stride;
  const int32_t slot = slot_ids[t];
  ST* dst = slot >= 0 ? cache + (int64_t)(slot / block_size) * cache_block_stride + (int64_t)(slot % block_size) * cache_row_stride : nullptr;
  // the two latents in turn: (source offset, length, weight, destination)
  for (int which = 0; which < 2; ++which) {
    const int64_t off = which ? kv_off : q_off, n = which ? kv_rank : q_rank;
    const float* w = which ? kv_w : q_w;
    ST* out = which ? dst : cq_out + t * q_rank;
    if (!out) break;
    float ss = 0.f;
    if (vec) {
      for (int64_t i = 4 * lane; i < n; i += 256) {
        const ST4 v = *reinterpret_cast<const ST4*>(p + off + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += A::to_float(v[e]) * A::to_float(v[e]);
      }
    } else {
      for (int64_t i = lane; i < n; i += 64) ss += A::to_float(p[off + i]) * A::to_float(p[off + i]);
    }
    const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)n + eps);
    if (vec) {
      for (int64_t i = 4 * lane; i < n; i += 256) {
        const ST4 v = *reinterpret_cast<const ST4*>(p + off + i);
        const f32x4 wv = *reinterpret_cast<const f32x4*>(w + i);
        ST4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = A::from_float(A::to_float(v[e]) * inv * wv[e]);
        *reinterpret_cast<ST4*>(out + i) = o;
      }
    } else {
      for (int64_t i = lane; i < n; i += 64) out[i] = A::from_float(A::to_float(p[off + i]) * inv * w[i]);
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Row form: one wave per (token, head).  Keys go by in groups of 64: lane l scores key lo + l (its own row of the
// cache against the query in LDS), the group's maximum and sum are wave reductions, then the lanes turn to the latent's
// columns (lane l owns columns l, l + 64, ...) and add the 64 rows, each weighted by its lane's p.  Serves float32 runs
// and layouts that are not 16-byte aligned; bfloat16 runs take the MFMA forms below.
// ---------------------------------------------------------------------------------------------------------------
constexpr int kMaxCols = HXM_MAX_LATENT / 64;

template <typename A>
__global__ __launch_bounds__(256) void latent_attn_rows_kernel(hxm_latent_attn_args a) {
  extern __shared__ float lds[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t total = (int64_t)a.n_tokens * a.n_heads;
  const bool live = (int64_t)blockIdx.x * 4 + wave < total;
  const int64_t item = live ? (int64_t)blockIdx.x * 4 + wave : total - 1;      // (a spare wave repeats the last row and stores nothing)
  const int32_t t = (int32_t)(item / a.n_heads), h = (int32_t)(item % a.n_heads);
  const int32_t R = a.kv_rank;
  float* q = lds + wave * R;
  const typename A::storage* qg = (const typename A::storage*)a.q + (int64_t)t * a.q_token_stride + (int64_t)h * a.q_head_stride;
  for (int i = lane; i < R; i += 64) q[i] = A::to_float(qg[i]) * a.scale;
  __syncthreads();
  const int32_t b = a.tok_seq[t];
  const int32_t pos = a.positions[t];
  const int32_t lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  const int32_t* table = a.block_table + a.cu_block_lens[b];
  const typename A::storage* cache = (const typename A::storage*)a.cache;
  constexpr int kVec = 16 / sizeof(typename A::storage);
  const bool vec = R % kVec == 0 && a.cache_row_stride % kVec == 0 && a.cache_block_stride % kVec == 0 &&
                   (reinterpret_cast<uintptr_t>(a.cache) & 15u) == 0;
  float m = -INFINITY, l = 0.f;
  float acc[kMaxCols];
#pragma unroll
  for (int k = 0; k < kMaxCols; ++k) acc[k] = 0.f;
  for (int32_t j0 = lo; j0 <= pos; j0 += 64) {
    const int32_t j = j0 + lane;
    const bool valid = j <= pos;
    int64_t off = 0;
    float s = -INFINITY;
    if (valid) {
      off = (int64_t)table[j / a.block_size] * a.cache_block_stride + (int64_t)(j % a.block_size) * a.cache_row_stride;
      const typename A::storage* c = cache + off;
      float d = 0.f;
      if (vec) {      // 16-byte loads of the row
        constexpr int N = 16 / sizeof(typename A::storage);
        typedef typename A::storage VecT __attribute__((ext_vector_type(N)));
        for (int i = 0; i < R; i += N) {
          const VecT v = *reinterpret_cast<const VecT*>(c + i);
#pragma unroll
          for (int e = 0; e < N; ++e) d += q[i + e] * A::to_float(v[e]);
        }
      } else {
        for (int i = 0; i < R; ++i) d += q[i] * A::to_float(c[i]);
      }
      s = d;
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float p = valid ? expf(s - m_new) : 0.f;
    const float corr = expf(m - m_new);      // (m = -inf on the first group: 0)
    l = l * corr + wave_sum(p);
    m = m_new;
#pragma unroll
    for (int k = 0; k < kMaxCols; ++k) acc[k] *= corr;
    const int n = min(64, pos - j0 + 1);
    for (int jj = 0; jj < n; ++jj) {
      const float pj = __shfl(p, jj, 64);
      const int64_t oj = __shfl(off, jj, 64);
      const typename A::storage* c = cache + oj;
#pragma unroll
      for (int k = 0; k < kMaxCols; ++k) {
        const int i = lane + 64 * k;
        if (i < R) acc[k] += pj * A::to_float(c[i]);
      }
    }
  }
  if (a.sinks) l += expf(a.sinks[h] - m);      // the sink: one more term of the denominator, without a value
  float g = 1.0f / l;
  if (a.gate_pre) {
    const float z = A::to_float(((const typename A::storage*)a.gate_pre)[(int64_t)t * a.gate_stride + h]);
    g = g / (1.0f + expf(-z));
  }
  typename A::storage* og = (typename A::storage*)a.out + (int64_t)t * a.out_token_stride + (int64_t)h * a.out_head_stride;
#pragma unroll
  for (int k = 0; k < kMaxCols; ++k) {
    const int i = lane + 64 * k;
    if (i < R && live) og[i] = A::from_float(acc[k] * g);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Tile form (bfloat16): one wave per 16 rows, a row being a (token, head) pair of ONE sequence's portion, heads fastest —
// sixteen heads of a decoded token, or a few tokens times a few heads.  All rows of a tile read the same keys, which go
// by in chunks of 32: S = Q C^T and O += P C are 16x16x32 MFMAs.  The chunk's rows come straight from the paged cache
// into the B operands of S (a lane's 16 bytes are 8 consecutive columns of one key's row); for O the same registers are
// written to the wave's LDS as they are (row-major image of the chunk, 16 bytes a write) and come back through the
// transposing LDS read (ds_read_b64_tr_b16: a lane gets one column of four rows) as B operands; P goes through LDS from
// the accumulator layout to the A layout.  Inside a chunk the 32 keys are summed in the order the transposing read
// delivers them — lane group g: keys 4g .. 4g+3, then 16+4g .. 16+4g+3 — in both operands.  No workgroup barriers: a wave
// shares nothing with its neighbours.
// ---------------------------------------------------------------------------------------------------------------
constexpr int kPStride = 36;       // u16 per row of P in LDS: 32 slots + 4

template <int KK>                  // ceil(kv_rank / 32), 1 .. 16
__global__ __launch_bounds__(256) void latent_attn_tile_kernel(hxm_latent_attn_args a, int tiles_per_seq, int waves_per_block) {
  extern __shared__ float lds[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (wave >= waves_per_block) return;
  const int n_splits = a.n_splits > 1 ? a.n_splits : 1;
  const int64_t witem = (int64_t)blockIdx.x * waves_per_block + wave;      // (sequence, row tile, key split), splits fastest
  if (witem >= (int64_t)a.n_seq * tiles_per_seq * n_splits) return;
  const int64_t item = witem / n_splits;
  const int split = (int)(witem % n_splits);
  const int b = (int)(item / tiles_per_seq), tile = (int)(item % tiles_per_seq);
  const int H = a.n_heads, R = a.kv_rank;
  const int q0 = a.q_cu[b];
  const int n_rows = (a.q_cu[b + 1] - q0) * H;
  if (tile * 16 >= n_rows) return;
  const int g = lane >> 4, c = lane & 15;
  const int R16 = (R + 15) / 16 * 16;
  const int RS = 2 * (KK * 32) + 32;      // bytes per row of the chunk's image (a key's columns, padded)
  char* img = reinterpret_cast<char*>(lds) + (size_t)wave * (32 * RS + 16 * kPStride * 2);
  u16* pl = reinterpret_cast<u16*>(img + 32 * RS);
  const u16* cache = (const u16*)a.cache;
  const int32_t* table = a.block_table + a.cu_block_lens[b];

  // the queries: lane (g, c) holds row c, columns 32 kk + 8 g .. + 7
  const int last_row = min(tile * 16 + 15, n_rows - 1);
  u16x8 qf[KK];
  {
    const int r = min(tile * 16 + c, n_rows - 1);
    const u16* qg = (const u16*)a.q + (int64_t)(q0 + r / H) * a.q_token_stride + (int64_t)(r % H) * a.q_head_stride;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const int col = 32 * kk + 8 * g;
      if (col < R) qf[kk] = *reinterpret_cast<const u16x8*>(qg + col);
      else qf[kk] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }
  // the rows this lane holds of S and O: 4 g + i
  int pos[4], lo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = tile * 16 + 4 * g + i;
    if (r < n_rows) {
      pos[i] = a.positions[q0 + r / H];
      lo[i] = a.window > 0 ? max(0, pos[i] - a.window + 1) : 0;
    } else {
      pos[i] = -1;      // sees nothing
      lo[i] = 0;
    }
  }
  // the keys any row of the tile sees: lane (., c) looks at row c, the sixteen are reduced by shuffles
  int k_min, k_max;
  {
    const int r = min(tile * 16 + c, last_row);
    const int pr = a.positions[q0 + r / H];
    k_max = pr;
    k_min = a.window > 0 ? max(0, pr - a.window + 1) : 0;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
      k_max = max(k_max, __shfl_xor(k_max, off, 64));
      k_min = min(k_min, __shfl_xor(k_min, off, 64));
    }
  }

  float m[4], l[4];
  f32x4 acc[KK * 2];
#pragma unroll
  for (int i = 0; i < 4; ++i) { m[i] = -1.0e30f; l[i] = 0.f; }
#pragma unroll
  for (int n = 0; n < KK * 2; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};

  // a key split takes a run of whole 32-key chunks of the tile's range (the last splits may get none)
  int k_begin = k_min, k_end = k_max;
  if (n_splits > 1) {
    const int chunks = (k_max - k_min + 32) / 32;
    const int per = (chunks + n_splits - 1) / n_splits;
    k_begin = k_min + split * per * 32;
    k_end = min(k_max, k_begin + per * 32 - 1);
  }
  const int bs = a.block_size;
  const int bshift = (bs & (bs - 1)) == 0 ? __ffs(bs) - 1 : -1;
  // half a chunk's rows, this lane's part: key 16 s + c, columns 32 kk + 8 g .. + 7
  auto fetch = [&](int key0, int s, u16x8 (&cf)[KK]) __attribute__((always_inline)) {
    const int key = min(key0 + 16 * s + c, k_max);        // (a key past the last one repeats it; masked below)
    const int page = bshift >= 0 ? key >> bshift : key / bs;
    const u16* row = cache + (int64_t)table[page] * a.cache_block_stride + (int64_t)(key - page * bs) * a.cache_row_stride;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const int col = 32 * kk + 8 * g;
      if (col < R) cf[kk] = *reinterpret_cast<const u16x8*>(row + col);
      else cf[kk] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  };
  // scores of half a chunk, and its rows into the image for the second product (row = key 16 s + c, the lane's eight
  // columns as they came)
  auto score = [&](int s, const u16x8 (&cf)[KK]) __attribute__((always_inline)) -> f32x4 {
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      v = Mfma<BF16>::mma(qf[kk], cf[kk], v);
      *reinterpret_cast<u16x8*>(img + (16 * s + c) * RS + (32 * kk + 8 * g) * 2) = cf[kk];
    }
    return v;
  };
  auto finish = [&](int key0, const f32x4 (&sc)[2]) __attribute__((always_inline)) {
    // softmax of the rows 4 g + i over this chunk (sc[s][i] is key key0 + 16 s + c)
    float p[2][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float mx = -INFINITY;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int key = key0 + 16 * s + c;
        const bool seen = key >= lo[i] && key <= pos[i];
        const float v = seen ? sc[s][i] * a.scale : -INFINITY;
        p[s][i] = v;
        mx = fmaxf(mx, v);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 1, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 2, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 4, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 8, 64));
      const float m_new = fmaxf(m[i], mx);
      const float corr = __expf(m[i] - m_new);
      float ps = 0.f;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        p[s][i] = __expf(p[s][i] - m_new);       // exp(-inf) = 0 for a key the row does not see
        ps += p[s][i];
      }
      ps += __shfl_xor(ps, 1, 64);
      ps += __shfl_xor(ps, 2, 64);
      ps += __shfl_xor(ps, 4, 64);
      ps += __shfl_xor(ps, 8, 64);
      l[i] = l[i] * corr + ps;
      m[i] = m_new;
#pragma unroll
      for (int n = 0; n < KK * 2; ++n) acc[n][i] *= corr;
      // key 16 s + c sits in slot 8 (c / 4) + c % 4 + 4 s of its row
      pl[(4 * g + i) * kPStride + 8 * (c >> 2) + (c & 3)] = BF16::from_float(p[0][i]);
      pl[(4 * g + i) * kPStride + 8 * (c >> 2) + (c & 3) + 4] = BF16::from_float(p[1][i]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // O += P C: A = P[row c][slots 8 g ..], B = the image's column 16 n + c at the keys of those slots
    u16x8 pf;
    {
      const u16x4 x0 = *reinterpret_cast<const u16x4*>(pl + c * kPStride + 8 * g);
      const u16x4 x1 = *reinterpret_cast<const u16x4*>(pl + c * kPStride + 8 * g + 4);
      pf = u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
    }
    const char* vrd = img + (4 * g + (c >> 2)) * RS + (c & 3) * 8;
#pragma unroll
    for (int n = 0; n < KK * 2; ++n) {
      {      // (column tiles past the latent's width read zeros of the image: no branch around an MFMA)
        const u16x4 x0 = lds_tr_read(vrd + n * 32);
        const u16x4 x1 = lds_tr_read(vrd + 16 * RS + n * 32);
        const u16x8 vf = u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
        acc[n] = Mfma<BF16>::mma(pf, vf, acc[n]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();      // the reads are done before the next chunk is written
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  {
    // two register sets: the next chunk's rows are on their way while this one is worked on
    u16x8 ca[2][KK], cb[2][KK];
    f32x4 sc[2];
    if (k_begin <= k_end) {
      fetch(k_begin, 0, ca[0]);
      fetch(k_begin, 1, ca[1]);
    }
    for (int key0 = k_begin; key0 <= k_end; key0 += 64) {
      const bool more = key0 + 32 <= k_end;
      if (more) {
        fetch(key0 + 32, 0, cb[0]);
        fetch(key0 + 32, 1, cb[1]);
      }
      sc[0] = score(0, ca[0]);
      sc[1] = score(1, ca[1]);
      finish(key0, sc);
      if (more) {
        if (key0 + 64 <= k_end) {
          fetch(key0 + 64, 0, ca[0]);
          fetch(key0 + 64, 1, ca[1]);
        }
        sc[0] = score(0, cb[0]);
        sc[1] = score(1, cb[1]);
        finish(key0 + 32, sc);
      }
    }
  }
  if (n_splits > 1) {
    // unnormalised partial result of this split: ws_o [item][split][16 rows][R16], ws_ml [item][split][16 rows][m, l]
    float* wo = a.ws_o + ((size_t)witem * 16) * R16;
    float* wml = a.ws_ml + (size_t)witem * 32;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * g + i;
      if (c == 0) {
        wml[2 * row] = m[i];
        wml[2 * row + 1] = l[i];
      }
#pragma unroll
      for (int n = 0; n < KK * 2; ++n) {
        const int col = 16 * n + c;
        if (col < R16) wo[(size_t)row * R16 + col] = acc[n][i];
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = tile * 16 + 4 * g + i;
    if (r >= n_rows) continue;
    const int t = q0 + r / H, h = r % H;
    float gsc = 1.0f / (a.sinks ? l[i] + expf(a.sinks[h] - m[i]) : l[i]);
    if (a.gate_pre) {
      const float z = BF16::to_float(((const u16*)a.gate_pre)[(int64_t)t * a.gate_stride + h]);
      gsc = gsc / (1.0f + __expf(-z));
    }
    u16* og = (u16*)a.out + (int64_t)t * a.out_token_stride + (int64_t)h * a.out_head_stride;
#pragma unroll
    for (int n = 0; n < KK * 2; ++n) {
      const int col = 16 * n + c;
      if (col < R) og[col] = BF16::from_float(acc[n][i] * gsc);
    }
  }
}

// The same for latents of more than 256 columns: no second register set for the rows on their way (the accumulators
// and the queries leave no room), a whole chunk in registers between its two products.
template <int KK>                  // ceil(kv_rank / 32), 9 .. 16
__global__ __launch_bounds__(256) void latent_attn_tile_wide_kernel(hxm_latent_attn_args a, int tiles_per_seq, int waves_per_block) {
  extern __shared__ float lds[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (wave >= waves_per_block) return;
  const int n_splits = a.n_splits > 1 ? a.n_splits : 1;
  const int64_t witem = (int64_t)blockIdx.x * waves_per_block + wave;      // (sequence, row tile, key split), splits fastest
  if (witem >= (int64_t)a.n_seq * tiles_per_seq * n_splits) return;
  const int64_t item = witem / n_splits;
  const int split = (int)(witem % n_splits);
  const int b = (int)(item / tiles_per_seq), tile = (int)(item % tiles_per_seq);
  const int H = a.n_heads, R = a.kv_rank;
  const int q0 = a.q_cu[b];
  const int n_rows = (a.q_cu[b + 1] - q0) * H;
  if (tile * 16 >= n_rows) return;
  const int g = lane >> 4, c = lane & 15;
  const int R16 = (R + 15) / 16 * 16;
  const int RS = 2 * (KK * 32) + 32;      // bytes per row of the chunk's image (a key's columns, padded)
  char* img = reinterpret_cast<char*>(lds) + (size_t)wave * (32 * RS + 16 * kPStride * 2);
  u16* pl = reinterpret_cast<u16*>(img + 32 * RS);
  const u16* cache = (const u16*)a.cache;
  const int32_t* table = a.block_table + a.cu_block_lens[b];

  // the queries: lane (g, c) holds row c, columns 32 kk + 8 g .. + 7
  const int last_row = min(tile * 16 + 15, n_rows - 1);
  u16x8 qf[KK];
  {
    const int r = min(tile * 16 + c, n_rows - 1);
    const u16* qg = (const u16*)a.q + (int64_t)(q0 + r / H) * a.q_token_stride + (int64_t)(r % H) * a.q_head_stride;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const int col = 32 * kk + 8 * g;
      if (col < R) qf[kk] = *reinterpret_cast<const u16x8*>(qg + col);
      else qf[kk] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }
  // the rows this lane holds of S and O: 4 g + i
  int pos[4], lo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = tile * 16 + 4 * g + i;
    if (r < n_rows) {
      pos[i] = a.positions[q0 + r / H];
      lo[i] = a.window > 0 ? max(0, pos[i] - a.window + 1) : 0;
    } else {
      pos[i] = -1;      // sees nothing
      lo[i] = 0;
    }
  }
  // the keys any row of the tile sees: lane (., c) looks at row c, the sixteen are reduced by shuffles
  int k_min, k_max;
  {
    const int r = min(tile * 16 + c, last_row);
    const int pr = a.positions[q0 + r / H];
    k_max = pr;
    k_min = a.window > 0 ? max(0, pr - a.window + 1) : 0;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
      k_max = max(k_max, __shfl_xor(k_max, off, 64));
      k_min = min(k_min, __shfl_xor(k_min, off, 64));
    }
  }

  float m[4], l[4];
  f32x4 acc[KK * 2];
#pragma unroll
  for (int i = 0; i < 4; ++i) { m[i] = -1.0e30f; l[i] = 0.f; }
#pragma unroll
  for (int n = 0; n < KK * 2; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};

  // a key split takes a run of whole 32-key chunks of the tile's range (the last splits may get none)
  int k_begin = k_min, k_end = k_max;
  if (n_splits > 1) {
    const int chunks = (k_max - k_min + 32) / 32;
    const int per = (chunks + n_splits - 1) / n_splits;
    k_begin = k_min + split * per * 32;
    k_end = min(k_max, k_begin + per * 32 - 1);
  }
  for (int key0 = k_begin; key0 <= k_end; key0 += 32) {
    f32x4 sc[2];
    u16x8 cf[2][KK];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int key = min(key0 + 16 * s + c, k_max);        // (a key past the last one repeats it; masked below)
      const u16* row = cache + (int64_t)table[key / a.block_size] * a.cache_block_stride +
                       (int64_t)(key % a.block_size) * a.cache_row_stride;
      sc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        const int col = 32 * kk + 8 * g;
        if (col < R) cf[s][kk] = *reinterpret_cast<const u16x8*>(row + col);
        else cf[s][kk] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
        sc[s] = Mfma<BF16>::mma(qf[kk], cf[s][kk], sc[s]);
      }
    }
    // the chunk's image for the second product: row = key 16 s + c, the lane's eight columns as they came
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
        *reinterpret_cast<u16x8*>(img + (16 * s + c) * RS + (32 * kk + 8 * g) * 2) = cf[s][kk];
    // softmax of the rows 4 g + i over this chunk (sc[s][i] is key key0 + 16 s + c)
    float p[2][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float mx = -INFINITY;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int key = key0 + 16 * s + c;
        const bool seen = key >= lo[i] && key <= pos[i];
        const float v = seen ? sc[s][i] * a.scale : -INFINITY;
        p[s][i] = v;
        mx = fmaxf(mx, v);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 1, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 2, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 4, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 8, 64));
      const float m_new = fmaxf(m[i], mx);
      const float corr = __expf(m[i] - m_new);
      float ps = 0.f;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        p[s][i] = __expf(p[s][i] - m_new);       // exp(-inf) = 0 for a key the row does not see
        ps += p[s][i];
      }
      ps += __shfl_xor(ps, 1, 64);
      ps += __shfl_xor(ps, 2, 64);
      ps += __shfl_xor(ps, 4, 64);
      ps += __shfl_xor(ps, 8, 64);
      l[i] = l[i] * corr + ps;
      m[i] = m_new;
#pragma unroll
      for (int n = 0; n < KK * 2; ++n) acc[n][i] *= corr;
      // key 16 s + c sits in slot 8 (c / 4) + c % 4 + 4 s of its row
      pl[(4 * g + i) * kPStride + 8 * (c >> 2) + (c & 3)] = BF16::from_float(p[0][i]);
      pl[(4 * g + i) * kPStride + 8 * (c >> 2) + (c & 3) + 4] = BF16::from_float(p[1][i]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // O += P C: A = P[row c][slots 8 g ..], B = the image's column 16 n + c at the keys of those slots
    u16x8 pf;
    {
      const u16x4 x0 = *reinterpret_cast<const u16x4*>(pl + c * kPStride + 8 * g);
      const u16x4 x1 = *reinterpret_cast<const u16x4*>(pl + c * kPStride + 8 * g + 4);
      pf = u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
    }
    const char* vrd = img + (4 * g + (c >> 2)) * RS + (c & 3) * 8;
#pragma unroll
    for (int n = 0; n < KK * 2; ++n) {
      {      // (column tiles past the latent's width read zeros of the image: no branch around an MFMA)
        const u16x4 x0 = lds_tr_read(vrd + n * 32);
        const u16x4 x1 = lds_tr_read(vrd + 16 * RS + n * 32);
        const u16x8 vf = u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
        acc[n] = Mfma<BF16>::mma(pf, vf, acc[n]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();      // the reads are done before the next chunk is written
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }

  if (n_splits > 1) {
    // unnormalised partial result of this split: ws_o [item][split][16 rows][R16], ws_ml [item][split][16 rows][m, l]
    float* wo = a.ws_o + ((size_t)witem * 16) * R16;
    float* wml = a.ws_ml + (size_t)witem * 32;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * g + i;
      if (c == 0) {
        wml[2 * row] = m[i];
        wml[2 * row + 1] = l[i];
      }
#pragma unroll
      for (int n = 0; n < KK * 2; ++n) {
        const int col = 16 * n + c;
        if (col < R16) wo[(size_t)row * R16 + col] = acc[n][i];
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = tile * 16 + 4 * g + i;
    if (r >= n_rows) continue;
    const int t = q0 + r / H, h = r % H;
    float gsc = 1.0f / (a.sinks ? l[i] + expf(a.sinks[h] - m[i]) : l[i]);
    if (a.gate_pre) {
      const float z = BF16::to_float(((const u16*)a.gate_pre)[(int64_t)t * a.gate_stride + h]);
      gsc = gsc / (1.0f + __expf(-z));
    }
    u16* og = (u16*)a.out + (int64_t)t * a.out_token_stride + (int64_t)h * a.out_head_stride;
#pragma unroll
    for (int n = 0; n < KK * 2; ++n) {
      const int col = 16 * n + c;
      if (col < R) og[col] = BF16::from_float(acc[n][i] * gsc);
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Group form (bfloat16, portions of prompts): a workgroup of four waves takes four consecutive row tiles (64 rows) of a
// sequence and ONE image of every 32-key chunk: each wave brings eight of the chunk's rows from the paged cache into
// LDS, then all four read their B operands of both products from there (16-byte reads for S, transposing reads for O).
// Against the tile form: a quarter of the global reads and LDS writes per wave, and no registers spent on the chunk.
// Two workgroup barriers a chunk (image complete / image free).  Used for latents of more than 256 columns.
// ---------------------------------------------------------------------------------------------------------------
template <int KK>
__global__ __launch_bounds__(256) void latent_attn_group_kernel(hxm_latent_attn_args a, int groups_per_seq) {
  extern __shared__ float lds[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t item = blockIdx.x;      // (sequence, group of four row tiles)
  const int b = (int)(item / groups_per_seq), grp = (int)(item % groups_per_seq);
  const int H = a.n_heads, R = a.kv_rank;
  const int q0 = a.q_cu[b];
  const int n_rows = (a.q_cu[b + 1] - q0) * H;
  if (grp * 64 >= n_rows) return;       // (the whole workgroup)
  const int tile = grp * 4 + wave;
  const bool live = tile * 16 < n_rows; // a wave without rows still brings its share of every chunk
  const int g = lane >> 4, c = lane & 15;
  const int RS = 2 * (KK * 32) + 32;    // bytes per row of the chunk's image (a key's columns, padded)
  char* img = reinterpret_cast<char*>(lds);
  u16* pl = reinterpret_cast<u16*>(img + 32 * RS) + wave * 16 * kPStride;
  const u16* cache = (const u16*)a.cache;
  const int32_t* table = a.block_table + a.cu_block_lens[b];
  // the image's columns past the latent's width stay zero (the loads below never touch them)
  for (int i = threadIdx.x; i < 2 * RS; i += 256) reinterpret_cast<u16x8*>(img)[i] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};

  u16x8 qf[KK];
  {
    const int r = min(tile * 16 + c, n_rows - 1);
    const u16* qg = (const u16*)a.q + (int64_t)(q0 + r / H) * a.q_token_stride + (int64_t)(r % H) * a.q_head_stride;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const int col = 32 * kk + 8 * g;
      if (col < R) qf[kk] = *reinterpret_cast<const u16x8*>(qg + col);
      else qf[kk] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }
  int pos[4], lo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = tile * 16 + 4 * g + i;
    if (r < n_rows) {
      pos[i] = a.positions[q0 + r / H];
      lo[i] = a.window > 0 ? max(0, pos[i] - a.window + 1) : 0;
    } else {
      pos[i] = -1;      // sees nothing
      lo[i] = 0;
    }
  }
  // the keys any row of the GROUP sees (the same in every wave): lane l looks at row 64 grp + l
  int k_min, k_max;
  {
    const int r = min(grp * 64 + lane, n_rows - 1);
    const int pr = a.positions[q0 + r / H];
    k_max = pr;
    k_min = a.window > 0 ? max(0, pr - a.window + 1) : 0;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      k_max = max(k_max, __shfl_xor(k_max, off, 64));
      k_min = min(k_min, __shfl_xor(k_min, off, 64));
    }
  }
  float m[4], l[4];
  f32x4 acc[KK * 2];
#pragma unroll
  for (int i = 0; i < 4; ++i) { m[i] = -1.0e30f; l[i] = 0.f; }
#pragma unroll
  for (int n = 0; n < KK * 2; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int bs = a.block_size;
  const int bshift = (bs & (bs - 1)) == 0 ? __ffs(bs) - 1 : -1;
  auto finish = [&](int key0, const f32x4 (&sc)[2]) __attribute__((always_inline)) {
    // softmax of the rows 4 g + i over this chunk (sc[s][i] is key key0 + 16 s + c)
    float p[2][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float mx = -INFINITY;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int key = key0 + 16 * s + c;
        const bool seen = key >= lo[i] && key <= pos[i];
        const float v = seen ? sc[s][i] * a.scale : -INFINITY;
        p[s][i] = v;
        mx = fmaxf(mx, v);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 1, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 2, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 4, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 8, 64));
      const float m_new = fmaxf(m[i], mx);
      const float corr = __expf(m[i] - m_new);
      float ps = 0.f;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        p[s][i] = __expf(p[s][i] - m_new);       // exp(-inf) = 0 for a key the row does not see
        ps += p[s][i];
      }
      ps += __shfl_xor(ps, 1, 64);
      ps += __shfl_xor(ps, 2, 64);
      ps += __shfl_xor(ps, 4, 64);
      ps += __shfl_xor(ps, 8, 64);
      l[i] = l[i] * corr + ps;
      m[i] = m_new;
#pragma unroll
      for (int n = 0; n < KK * 2; ++n) acc[n][i] *= corr;
      // key 16 s + c sits in slot 8 (c / 4) + c % 4 + 4 s of its row
      pl[(4 * g + i) * kPStride + 8 * (c >> 2) + (c & 3)] = BF16::from_float(p[0][i]);
      pl[(4 * g + i) * kPStride + 8 * (c >> 2) + (c & 3) + 4] = BF16::from_float(p[1][i]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // O += P C: A = P[row c][slots 8 g ..], B = the image's column 16 n + c at the keys of those slots
    u16x8 pf;
    {
      const u16x4 x0 = *reinterpret_cast<const u16x4*>(pl + c * kPStride + 8 * g);
      const u16x4 x1 = *reinterpret_cast<const u16x4*>(pl + c * kPStride + 8 * g + 4);
      pf = u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
    }
    const char* vrd = img + (4 * g + (c >> 2)) * RS + (c & 3) * 8;
#pragma unroll
    for (int n = 0; n < KK * 2; ++n) {
      {      // (column tiles past the latent's width read zeros of the image: no branch around an MFMA)
        const u16x4 x0 = lds_tr_read(vrd + n * 32);
        const u16x4 x1 = lds_tr_read(vrd + 16 * RS + n * 32);
        const u16x8 vf = u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
        acc[n] = Mfma<BF16>::mma(pf, vf, acc[n]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();      // the reads are done before the next chunk is written
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  __syncthreads();      // the zeroed image
  for (int key0 = k_min; key0 <= k_max; key0 += 32) {
    // this wave's eight rows of the chunk: key0 + 8 wave + kq, a lane brings eight columns
#pragma unroll
    for (int kq = 0; kq < 8; ++kq) {
      const int key = min(key0 + 8 * wave + kq, k_max);      // (a key past the last one repeats it; masked in the softmax)
      const int page = bshift >= 0 ? key >> bshift : key / bs;
      const u16* row = cache + (int64_t)table[page] * a.cache_block_stride + (int64_t)(key - page * bs) * a.cache_row_stride;
      for (int col = lane * 8; col < R; col += 512)
        *reinterpret_cast<u16x8*>(img + (8 * wave + kq) * RS + col * 2) = *reinterpret_cast<const u16x8*>(row + col);
    }
    __syncthreads();      // the image is complete
    if (live) {
      f32x4 sc[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        sc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
          sc[s] = Mfma<BF16>::mma(qf[kk], *reinterpret_cast<const u16x8*>(img + (16 * s + c) * RS + (32 * kk + 8 * g) * 2), sc[s]);
      }
      finish(key0, sc);
    }
    __syncthreads();      // every wave is done with the image
  }
  if (!live) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = tile * 16 + 4 * g + i;
    if (r >= n_rows) continue;
    const int t = q0 + r / H, h = r % H;
    float gsc = 1.0f / (a.sinks ? l[i] + expf(a.sinks[h] - m[i]) : l[i]);
    if (a.gate_pre) {
      const float z = BF16::to_float(((const u16*)a.gate_pre)[(int64_t)t * a.gate_stride + h]);
      gsc = gsc / (1.0f + __expf(-z));
    }
    u16* og = (u16*)a.out + (int64_t)t * a.out_token_stride + (int64_t)h * a.out_head_stride;
#pragma unroll
    for (int n = 0; n < KK * 2; ++n) {
      const int col = 16 * n + c;
      if (col < R) og[col] = BF16::from_float(acc[n][i] * gsc);
    }
  }
}

constexpr int64_t kTileWaves = 2048;      // what the tile form deals a launch of few rows to: 8 waves a CU

// ---------------------------------------------------------------------------------------------------------------
// Wide form (bfloat16, portions of prompts, latents of 64 KK columns, pages of whole 16-row groups): a workgroup of four waves takes
// 128 rows, 32 a wave, and goes over the keys in tiles of 64 whose rows go straight from the paged cache to LDS, the next tile's
// while this one is worked on.  The products are 32 x 32 x 16 and swapped, S^T = C Q^T and O^T += C^T P^T: a row of the softmax is a
// lane, its weights go into the second product from the registers they were made in.  Both products read the one image: 16-byte
// chunk x of row r sits at x ^ swz(r), with the row's two low bits above its next two, so that the 16 rows of one pass of a
// 16-byte read as well as the four rows of a transposing read fall into different banks.
// The tile and group forms read a row from LDS (or memory) once per 16 x 16 x 32 product; here a byte feeds twice the products.  A
// lane holds 48 KK registers of queries and accumulators: two waves a SIMD up to 192 columns; wider latents take the form below.
// (No register may spill here: the waits for scratch would be waits for the tile on its way.)
// A row's weights refer to its largest score so far, which costs a pass over the accumulators for nearly every tile.  (Left up to 2^8
// behind it, 64 columns took 35 us instead of 39, and results were off by 3 % more: the largest weights were rounded to bfloat16
// instead of being 1.)
// Measured, 4 portions of 797 - 1151 tokens, 32 heads: 64 columns 134 us in the tile form, 39 here, 128 columns 209 and 60, 192
// columns 393 and 84.  256 columns, 16 heads 70 us in this form, 65 in the one below; 320 columns 120 and 76.
// ---------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ f32x16 mma32(u16x8 a, u16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

template <int KK>
__global__ __launch_bounds__(256, 2) void latent_attn_wide_kernel(hxm_latent_attn_args a) {
  constexpr int R = 64 * KK, KT = 64, TQ = 128, KS = R / 16, NDB = R / 32, RS = 2 * R, L = R / 8, IMG = KT * RS;
  constexpr bool FULL = RS % 256 == 0;       // a row is whole bank rows (256 bytes): 16 rows need 16 places, else 8 of each parity
  extern __shared__ __attribute__((aligned(256))) char smem_w[];       // [2][64 rows]
  auto swz = [](int row) { return FULL ? ((row & 3) << 2 | (row >> 2 & 3)) : ((row >> 1 & 1) << 2 | (row >> 2 & 3)); };
  typedef __attribute__((address_space(4))) const int32_t c_i32;       // (uniform indices: through the scalar cache)
  c_i32* q_cu = (c_i32*)a.q_cu;
  const int H = a.n_heads;
  int b, tile, q0, n_rows;
  if (!find_row_tile<TQ>(q_cu, a.n_seq, H, blockIdx.x, b, tile, q0, n_rows)) return;      // spare slot (the grid is an upper bound)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = lane & 31, hi = lane >> 5;
  // row tiles end with the portion: a partial one is the first, with the fewest keys.  Rows below 0 do not exist.
  const int row0_wg = n_rows - ((n_rows + TQ - 1) / TQ - tile) * TQ, row0 = row0_wg + 32 * wave;
  const int r = max(row0 + c, 0), tok = r / H, head = r % H;
  auto first_key = [&](int p) { return a.window > 0 ? max(0, p - a.window + 1) : 0; };
  const int pos = a.positions[q0 + tok], lo = first_key(pos);
  // what the rows of the wave see, and any row of the workgroup (every wave looks at all of them: no order of the positions is assumed)
  const int wpos0 = wave_min_int(pos), wpos1 = wave_max_int(pos), wlo0 = wave_min_int(lo), wlo1 = wave_max_int(lo);
  int k_first, k_last;
  {
    const int p0 = a.positions[q0 + max(row0_wg + lane, 0) / H], p1 = a.positions[q0 + max(row0_wg + 64 + lane, 0) / H];
    k_first = wave_min_int(min(first_key(p0), first_key(p1)));
    k_last = wave_max_int(max(p0, p1));
  }
  const bool live = row0 + 31 >= 0;
  const int t_first = k_first / KT, t_last = k_last < 0 ? t_first - 1 : k_last / KT;      // (positions below 0 see nothing)

  const u16* cache = (const u16*)a.cache;
  c_i32* table = (c_i32*)(a.block_table + ((c_i32*)a.cu_block_lens)[b]);
  const int bs = a.block_size, bshift = (bs & (bs - 1)) == 0 ? __ffs(bs) - 1 : -1;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem_w;
  // Wave w brings keys 16 w .. of a tile (one page): 16 L chunks, 64 an instruction.  What lies in front of the first key that some row
  // sees, or behind the last, is not touched (its page may be gone): rows there repeat that key, masked.
  constexpr int NL = 16 * L / 64;
  auto bring = [&](int t, int img) __attribute__((always_inline)) {
    const int key0 = min(max(t * KT + 16 * wave, k_first & ~15), k_last), r_min = k_first - key0, r_max = k_last - key0;
    const int page = bshift >= 0 ? key0 >> bshift : key0 / bs;
    const u16* base = cache + (int64_t)table[page] * a.cache_block_stride + (int64_t)(key0 - page * bs) * a.cache_row_stride;
    const uint32_t to = lds0 + (uint32_t)(img * IMG + 16 * wave * RS);
    uint32_t ln = (uint32_t)lane;
    asm volatile("" : "+v"(ln));             // (worked out anew every time: kept, the addresses would push the queries out of registers)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    // (m0, the LDS address of the transfer, is a reserved register: nothing else in this kernel uses it)
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const int rr = (int)((64u * j + ln) / L), ch = (int)((64u * j + ln) % L);
      const uint32_t off = (uint32_t)max(min(rr, r_max), r_min) * (uint32_t)(2 * a.cache_row_stride) + 16u * (uint32_t)(ch ^ swz(rr));
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(__builtin_amdgcn_readfirstlane(to + 1024u * j)) : "memory", "m0");
    }
#pragma clang diagnostic pop
  };
  if (t_first <= t_last) bring(t_first, 0);
  u16x8 qf[KS];                              // the queries (B operand): row c, columns 16 ks + 8 hi ..
  {
    const u16* qg = (const u16*)a.q + (int64_t)(q0 + tok) * a.q_token_stride + (int64_t)head * a.q_head_stride + 8 * hi;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const u16x8*>(qg + 16 * ks);
    // (they are there before the loop: a wait for them inside it would be one for the tile on its way)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[ks]));
  }
  constexpr float kLog2e = 1.4426950408889634f;
  float scale2 = a.scale * kLog2e;
  if (scale2 < 0.f) {                        // (a maximum of scores is one of scaled scores where the scale is positive)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] ^= (u16)0x8000;
  }
  scale2 = fabsf(scale2) < 1e-30f ? 1e-30f : fabsf(scale2);      // (not fmaxf: what is not a number stays so)

  f32x16 acc[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
  float m = HX_NEG_BIG, l = 0.f;
  // Reads of rows: chunk 2 ks + hi of row c.  The swizzle touches the low four bits of a chunk (three where rows are not whole
  // bank rows): ks = NP x + y sits at x rows' worth of these and y bit by bit beside the place of ks = 0.
  constexpr int NP = FULL ? 8 : 4;
  const uint32_t kp0 = lds0 + (uint32_t)(c * RS + 16 * (hi ^ swz(c)));
  // Transposing reads: lane 4 q + p of every 16 lanes brings row 4 hi + q (and the row 8 below it), columns 16 half + 4 p .. of a
  // block of 32: chunks 4 db .. + 3, db = NB x + y the same way.
  constexpr int NB = FULL ? 4 : 2;
  uint32_t vp0, vp1;
  {
    const int q = (lane & 15) >> 2, p = lane & 3, x = 2 * ((lane >> 4) & 1) + (p >> 1);
    vp0 = lds0 + (uint32_t)((4 * hi + q) * RS + 16 * (x ^ swz(4 * hi + q)) + 8 * (p & 1));
    vp1 = lds0 + (uint32_t)((4 * hi + q + 8) * RS + 16 * (x ^ swz(4 * hi + q + 8)) + 8 * (p & 1));
  }
  auto row_read = [](uint32_t at) __attribute__((always_inline)) {
    return *reinterpret_cast<__attribute__((address_space(3))) const u16x8*>((uintptr_t)at);
  };
  auto tr_read = [](uint32_t at) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) hx_s16x4_t lds_s4;
    return __builtin_bit_cast(u16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(uintptr_t)at));
  };
  // 32 keys from key0 on, rows kt of the image (all 64 of a tile at once would not leave the registers for 512 columns)
  auto step = [&](int key0, uint32_t kt) __attribute__((always_inline)) {
    uint32_t kp = kp0, va = vp0, vb = vp1;
    asm volatile("" : "+v"(kp), "+v"(va), "+v"(vb));      // (their sums are made where they are read, not kept in registers)
    f32x16 s;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) s = mma32(row_read((kp ^ (32u * (ks % NP))) + kt + 32u * NP * (ks / NP)), qf[ks], s);
    // (reads stay a few products ahead)
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
    for (int i = 0; i < KS - 4; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
    const int key_l = key0 + 4 * hi;         // element e: key key_l + (e & 3) + 8 (e >> 2)
    float mx = HX_NEG_BIG;
    if (key0 + 31 <= wpos0 && key0 >= wlo1) {              // every row of the wave sees all of them
#pragma unroll
      for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[e]);
    } else {
      const int last = pos - key_l, first = lo - key_l;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int k = (e & 3) + 8 * (e >> 2);
        if (k > last || k < first) s[e] = -INFINITY;
        mx = fmaxf(mx, s[e]);
      }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    // (the weights always refer to the largest score so far: its own is then 1, which no rounding to bfloat16 touches)
    const float m_new = fmaxf(m, mx * scale2);
    if (__builtin_amdgcn_ballot_w64(m_new > m)) {
      const float alpha = fast_exp2(m - m_new);
      l *= alpha;
#pragma unroll
      for (int i = 0; i < NDB; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] *= alpha;
      m = m_new;
    }
    u16x8 pf[2];
    float pa = 0.f, pb = 0.f;
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
      const float e0 = fast_exp2(__builtin_fmaf(s[e], scale2, -m)), e1 = fast_exp2(__builtin_fmaf(s[e + 1], scale2, -m));
      pa += e0;
      pb += e1;
      pf[e >> 3][e & 7] = BF16::from_float(e0);
      pf[e >> 3][(e & 7) + 1] = BF16::from_float(e1);
    }
    l += pa + pb;
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2) {
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        const uint32_t at = kt + 16u * k2 * RS + 64u * NB * (db / NB);
        const u16x4 x0 = tr_read((va ^ (64u * (db % NB))) + at), x1 = tr_read((vb ^ (64u * (db % NB))) + at);
        acc[db] = mma32(u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]}, pf[k2], acc[db]);
      }
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
    for (int i = 0; i < 2 * NDB - 2; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
  };
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int t = t_first; t <= t_last; ++t) {
    const int img = (t - t_first) & 1;
    if (t < t_last) bring(t + 1, img ^ 1);
#pragma unroll 1
    for (int key0 = t * KT; key0 < t * KT + KT; key0 += 32)
      if (live && key0 <= wpos1 && key0 + 31 >= wlo0) step(key0, (uint32_t)(img * IMG + (key0 - t * KT) * RS));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this wave's part of the next tile is there
    __syncthreads();                                       // everybody's is, and this one has been read
  }
  if (!live) return;
  // out, through LDS (the images are free): whole rows a store.  O[row c][column 32 db + 8 (e >> 2) + 4 hi + (e & 3)]
  float total = l + __shfl_xor(l, 32, 64);
  if (a.sinks) total += fast_exp2(a.sinks[head] * kLog2e - m);      // the sink: one more term, without a value
  float gsc = 1.0f / total;
  if (a.gate_pre) {
    const float z = BF16::to_float(((const u16*)a.gate_pre)[(int64_t)(q0 + tok) * a.gate_stride + head]);
    gsc = gsc / (1.0f + __expf(-z));
  }
  char* ob = smem_w + wave * 32 * RS;
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4) {         // 8-byte slot 8 db + 2 e4 + hi of row c, turned by the row within its 128 bytes
      u16x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = BF16::from_float(acc[db][4 * e4 + i] * gsc);
      *reinterpret_cast<u16x4*>(ob + c * RS + (((8 * db + 2 * e4 + hi) ^ (c & 15)) << 3)) = o;
    }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int j = 0; j < 2 * NL; ++j) {
    const int rl = (64 * j + lane) / L, ch = (64 * j + lane) % L, ro = row0 + rl;
    // slots 2 ch, 2 ch + 1 of row rl sit in chunk ch ^ (rl' >> 1), in turned order when rl' is odd (rl' = rl mod 16)
    u16x8 v = *reinterpret_cast<const u16x8*>(ob + rl * RS + 16 * (ch ^ ((rl & 15) >> 1)));
    if (rl & 1) v = u16x8{v[4], v[5], v[6], v[7], v[0], v[1], v[2], v[3]};
    if (ro >= 0) *reinterpret_cast<u16x8*>((u16*)a.out + (int64_t)(q0 + ro / H) * a.out_token_stride + (int64_t)(ro % H) * a.out_head_stride + 8 * ch) = v;
  }
}

// The same for wider latents (64 KK columns): four waves of 16 rows, 16 x 16 x 32 products — a row's queries and
// accumulators are 192 registers a lane at 512 columns, two waves a SIMD.  A byte from LDS feeds half the products of the form
// above, but nothing is full (matrix cores 32 % of the time, vector ALU 39, LDS 30): a wave goes through scores, softmax and values in
// turn, waits for a quarter of its time, and there are two waves a SIMD.  Tiles of 32 keys and 64 rows: two workgroups a CU, one working while the other brings queries in or results
// out.  Also the form for few rows (short portions; single tokens of more than 32 heads, those of fewer are latent_step.hip's): the keys of a row tile are then dealt to several
// workgroups (wide_plan), each writes its rows' sums, maximum and weight, and the kernel below merges them.
// Measured, 4 portions of 797 - 1151 tokens, 32 heads, 512 columns: 861 us in the group form, 190 us here (670 TFLOP/s; 240 while the
// compiler had every read of a key waited for at once, 220 with addresses of the loads worked out lane by lane); 256 columns, 16
// heads 268 and 64 us, 320 columns 396 and 68.  32 tokens of 301 - 1747 keys, 32 heads, 512 columns under a window of 512: 31 us and
// 30 to merge in the tile form, 18 and 4.5 here (15.6 in all in latent_step.hip).
// (Thirty-two rows a wave, one wave a SIMD, with weights as sums of two bfloat16 numbers instead of a pass over the 256 accumulators:
// 245 us where this form took 253; the second set of products meets the card's power limit.)
// Row r of sixteen has its chunks at x ^ swz(r): rows r and 15 - r share a 32-byte place (their
// chunks turned), so that a pass of a 16-byte read (rows 0-3 and 12-15 of one chunk, 4-11 of the next) and a transposing read
// (eight rows, 32 bytes each) both reach every bank once.
template <int KK, bool FINE, int KG>      // FINE: every tile's weights refer to their own largest score; KG: groups of four waves, which share the keys
__global__ __launch_bounds__(256 * KG, 2) void latent_attn_wide16_kernel(hxm_latent_attn_args a, int tiles_per_seq) {
  constexpr int R = 64 * KK, KT = 32, TQ = 64, KPW = 8, KS = R / 32, NDB = R / 16, RS = 2 * R, L = R / 8, IMG = KT * RS;
  constexpr bool FULL = RS % 256 == 0;       // rows of whole bank rows: 16 places of a chunk, else 8 for each parity of the row
  extern __shared__ __attribute__((aligned(256))) char smem_w[];       // [KG][2][32 rows]
  auto swz = [](int row) {
    if (FULL) return (row & 15) < 8 ? 2 * (row & 7) : 31 - 2 * (row & 15);
    const int h = (row & 15) >> 1;
    return h < 4 ? 2 * h : 15 - 2 * h;
  };
  typedef __attribute__((address_space(4))) const int32_t c_i32;       // (uniform indices: through the scalar cache)
  c_i32* q_cu = (c_i32*)a.q_cu;
  const int H = a.n_heads;
  const int n_splits = FINE && a.n_splits > 1 ? a.n_splits : 1, split = n_splits > 1 ? (int)(blockIdx.x % n_splits) : 0;
  int b, tile, q0, n_rows;
  if (!find_row_tile<TQ>(q_cu, a.n_seq, H, (int)(n_splits > 1 ? blockIdx.x / n_splits : blockIdx.x), b, tile, q0, n_rows)) return;      // spare slot (the grid is an upper bound)
  const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3), lane = threadIdx.x & 63;
  const int group = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;      // takes every KG-th tile of keys
  const int c = lane & 15, g = lane >> 4;
  const int row0_wg = n_rows - ((n_rows + TQ - 1) / TQ - tile) * TQ, row0 = row0_wg + 16 * wave;
  const int r = max(row0 + c, 0), tok = r / H, head = r % H;
  auto first_key = [&](int p) { return a.window > 0 ? max(0, p - a.window + 1) : 0; };
  const int pos = a.positions[q0 + tok], lo = first_key(pos);
  const int wpos0 = wave_min_int(pos), wpos1 = wave_max_int(pos), wlo0 = wave_min_int(lo), wlo1 = wave_max_int(lo);
  static_assert(TQ == 64, "a lane looks at one row of the workgroup");
  const int p_wg = a.positions[q0 + max(row0_wg + lane, 0) / H];
  const int k_first = wave_min_int(first_key(p_wg)), k_last = wave_max_int(p_wg);
  const bool live = row0 + 15 >= 0;
  int t_first = k_first / KT, t_last = k_last < 0 ? t_first - 1 : k_last / KT;      // (positions below 0 see nothing)
  if (n_splits > 1) {                        // this split's run of tiles (the last splits may get none)
    const int per = (t_last - t_first + n_splits) / n_splits;
    t_first += split * per;
    t_last = min(t_last, t_first + per - 1);
  }

  const u16* cache = (const u16*)a.cache;
  c_i32* table = (c_i32*)(a.block_table + ((c_i32*)a.cu_block_lens)[b]);
  const int bs = a.block_size, bshift = (bs & (bs - 1)) == 0 ? __ffs(bs) - 1 : -1;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem_w + (uint32_t)(group * 2 * IMG);
  // Wave w brings keys 8 w .. of a tile (one page): 8 L chunks, 64 an instruction; none in front of the first or behind the last, as above.
  constexpr int NL = KPW * L / 64;
  const uint32_t row_bytes = (uint32_t)(2 * a.cache_row_stride);
  auto bring = [&](int t, int img) __attribute__((always_inline)) {
    const int key0 = min(max(t * KT + KPW * wave, k_first & ~(KPW - 1)), k_last), r_min = k_first - key0, r_max = k_last - key0;
    const int page = bshift >= 0 ? key0 >> bshift : key0 / bs;
    const u16* base = cache + (int64_t)table[page] * a.cache_block_stride + (int64_t)(key0 - page * bs) * a.cache_row_stride;
    const uint32_t to = lds0 + (uint32_t)(img * IMG + KPW * wave * RS);
    uint32_t ln = (uint32_t)lane;
    asm volatile("" : "+v"(ln));             // (worked out anew every time: kept, the addresses would push the queries out of registers)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    // (m0, the LDS address of the transfer, is a reserved register: nothing else in this kernel uses it)
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      uint32_t off;
      if constexpr (L == 64) {               // a row a load: nothing of it differs from lane to lane but the column
        off = (16u * ln ^ 16u * (uint32_t)swz(KPW * wave + j)) + (uint32_t)max(min(j, r_max), r_min) * row_bytes;
      } else {
        // (swz of row 8 wave + rr)
        const uint32_t rr = (64u * j + ln) / L, ch = 64u * j + ln - rr * L, turned = wave & 1 ? (FULL ? 15u : 7u) : 0u;
        off = (uint32_t)max(min((int)rr, r_max), r_min) * row_bytes + 16u * (ch ^ (FULL ? 2u * rr : rr & 6u) ^ turned);
      }
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(__builtin_amdgcn_readfirstlane(to + 1024u * j)) : "memory", "m0");
    }
#pragma clang diagnostic pop
  };
  if (t_first + group <= t_last) bring(t_first + group, 0);
  u16x8 qf[KS];                              // the queries (B operand): row c, columns 32 ks + 8 g ..
  {
    const u16* qg = (const u16*)a.q + (int64_t)(q0 + tok) * a.q_token_stride + (int64_t)head * a.q_head_stride + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const u16x8*>(qg + 32 * ks);
    // (they are there before the loop: a wait for them inside it would be one for the tile on its way)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[ks]));
  }
  constexpr float kLog2e = 1.4426950408889634f;
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
  // Reads of rows: chunk 4 ks + g of row c; the swizzle touches the low four (three) bits of a chunk, ks = NP x + y.  Transposing
  // reads: lane 4 q + p of a group of 16 brings row 4 g + q (and the row 16 below it: the same place), columns 16 db + 4 p ..:
  // chunk 2 db + p / 2, db = 2 NP x + y.
  constexpr int NP = FULL ? 4 : 2;
  const uint32_t kp0 = lds0 + (uint32_t)(c * RS + 16 * (g ^ swz(c)));
  const uint32_t vp0 = lds0 + (uint32_t)((4 * g + (c >> 2)) * RS + 16 * (((c & 3) >> 1) ^ swz(4 * g + (c >> 2))) + 8 * (c & 1));
  auto row_read = [](uint32_t at) __attribute__((always_inline)) {
    return *reinterpret_cast<__attribute__((address_space(3))) const u16x8*>((uintptr_t)at);
  };
  auto tr_read = [](uint32_t at) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) hx_s16x4_t lds_s4;
    return __builtin_bit_cast(u16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(uintptr_t)at));
  };
  // 32 keys from key0 on, rows kt of the image
  auto step = [&](int key0, uint32_t kt) __attribute__((always_inline)) {
    uint32_t kp = kp0 + kt, va = vp0 + kt;
    asm volatile("" : "+v"(kp), "+v"(va));   // (their sums are made where they are read, not kept in registers)
    // Rows of the keys, kAhead of them on their way.  The order is laid down product by product: left to the compiler, group barriers
    // or not, every read was waited for where it stood (LDS answers after some 150 cycles, a product takes 16).
    constexpr int kAhead = 2 * KS < 8 ? 2 * KS : 8;
    f32x4 s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) s[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto key_read = [&](int i) __attribute__((always_inline)) {
      return row_read((kp ^ (64u * (i / 2 % NP))) + 16u * (i & 1) * RS + 64u * NP * (i / 2 / NP));
    };
    u16x8 kf[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) kf[i] = key_read(i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i) {
      s[i & 1] = Mfma<BF16>::mma(kf[i % kAhead], qf[i / 2], s[i & 1]);
      if (i + kAhead < 2 * KS) kf[i % kAhead] = key_read(i + kAhead);
      __builtin_amdgcn_sched_barrier(0);
    }
    const int key_l = key0 + 4 * g;          // element e of half u: key key_l + 16 u + e
    float mx = HX_NEG_BIG;
    if (key0 + 31 <= wpos0 && key0 >= wlo1) {              // every row of the wave sees all of them
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, s[e >> 2][e & 3]);
    } else {
      const int last = pos - key_l, first = lo - key_l;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int k = 16 * (e >> 2) + (e & 3);
        if (k > last || k < first) s[e >> 2][e & 3] = -INFINITY;
        mx = fmaxf(mx, s[e >> 2][e & 3]);
      }
    }
    mx = groups_max(mx);
    // The weights refer to the largest score so far, as above — or, in launches of few rows, to the largest of these 32 keys, and what
    // they add is scaled behind the products: the tile form deals such a launch's keys to more waves, each with a largest score that
    // weighs exactly 1 (32 tokens of 301 - 1747 keys, 2-norm of the error over the result: 1.909e-3 there, 1.933e-3 with its own splits' largest
    // scores here, 1.900e-3 with every 32 keys').
    float m_ref = mx * scale2;
    asm("" : "+v"(m_ref));                   // (rounded: left inside a difference below it would not be m_new's number)
    const float m_new = fmaxf(m, m_ref), alpha = fast_exp2(m - m_new), beta = fast_exp2(m_ref - m_new);
    if constexpr (FINE) {
      l *= alpha;
    } else {
      m_ref = m_new;
      if (__builtin_amdgcn_ballot_w64(m_new > m)) {
        l *= alpha;
#pragma unroll
        for (int i = 0; i < NDB; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][e] *= alpha;
      }
    }
    m = m_new;
    u16x8 pf;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float p = fast_exp2(__builtin_fmaf(s[e >> 2][e & 3], scale2, -m_ref));
      l = FINE ? __builtin_fmaf(p, beta, l) : l + p;
      pf[e] = BF16::from_float(p);
    }
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      const uint32_t at = (va ^ (32u * (db % (2 * NP)))) + 64u * NP * (db / (2 * NP));
      const u16x4 x0 = tr_read(at), x1 = tr_read(at + 16u * RS);
      const u16x8 x = u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
      if constexpr (FINE) {
        const f32x4 o = Mfma<BF16>::mma(x, pf, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[db][e] = __builtin_fmaf(o[e], beta, acc[db][e] * alpha);
      } else {
        acc[db] = Mfma<BF16>::mma(x, pf, acc[db]);
      }
    }
    constexpr int kAheadV = NDB < 6 ? NDB : 6;
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kAheadV, 0);
#pragma unroll
    for (int i = 0; i < NDB - kAheadV; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kAheadV, 0);
  };
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int t0 = t_first; t0 <= t_last; t0 += KG) {
    const int t = t0 + group, img = (t0 - t_first) / KG & 1;
    if (t + KG <= t_last) bring(t + KG, img ^ 1);
    if (live && t <= t_last && t * KT <= wpos1 && t * KT + KT - 1 >= wlo0) step(t * KT, (uint32_t)(img * IMG));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this wave's part of the next tile is there
    __syncthreads();                                       // everybody's is, and this one has been read
  }
  // Two groups: each hands the other half of its columns and finishes the rest.  (One tile: the first group has it all.)
  const bool two = KG > 1 && t_last > t_first;
  if constexpr (KG > 1) {
    if (two) {
      f32x4* part = reinterpret_cast<f32x4*>(smem_w) + wave * NDB * 64 + lane;
      float2* ml = reinterpret_cast<float2*>(smem_w + 4 * NDB * 1024) + wave * 128 + lane;
      auto hand = [&](auto first) __attribute__((always_inline)) {      // (first: the first column block that the other group finishes)
#pragma unroll
        for (int i = first; i < first + NDB / 2; ++i) part[i * 64] = acc[i];
      };
      if (group) hand(std::integral_constant<int, 0>());
      else hand(std::integral_constant<int, NDB / 2>());
      ml[64 * group] = float2{m, l};
      __syncthreads();
      const float2 o = ml[64 * (1 - group)];
      const float top = fmaxf(m, o.x), mine = fast_exp2(m - top), theirs = fast_exp2(o.x - top);
      l = __builtin_fmaf(l, mine, o.y * theirs);
      m = top;
      auto take = [&](auto first) __attribute__((always_inline)) {
#pragma unroll
        for (int i = first; i < first + NDB / 2; ++i) {
          const f32x4 x = part[i * 64];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][e] = __builtin_fmaf(acc[i][e], mine, x[e] * theirs);
        }
      };
      if (group) take(std::integral_constant<int, NDB / 2>());
      else take(std::integral_constant<int, 0>());
      __syncthreads();                                     // (results go where these came from)
    } else if (group) {
      return;
    }
  }
  auto finishes = [&](int db) { return !two || (db >= NDB / 2) == (group != 0); };
  if (!live && !two) return;
  // out, through LDS (the images are free): whole rows a store.  O[row c][column 16 db + 4 g + e]
  float total = l + __shfl_xor(l, 16, 64);
  total += __shfl_xor(total, 32, 64);
  if (n_splits > 1) {
    // what this split adds to a row, not normalised: ws_o [sequence][row][split][R], ws_ml [..][split][maximum (log2), sum]
    if (row0 + c >= 0 && row0 + c < tiles_per_seq * 16) {      // (rows past max_q_len tokens have no place)
      const size_t at = ((size_t)b * tiles_per_seq * 16 + (row0 + c)) * n_splits + split;
      float* wo = a.ws_o + at * R + 4 * g;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
        if (finishes(db)) *reinterpret_cast<f32x4*>(wo + 16 * db) = acc[db];
      if (g == 0 && group == 0) {
        a.ws_ml[2 * at] = m;
        a.ws_ml[2 * at + 1] = total;
      }
    }
    return;
  }
  if (a.sinks) total += fast_exp2(a.sinks[head] * kLog2e - m);      // the sink: one more term, without a value
  float gsc = 1.0f / total;
  if (a.gate_pre) {
    const float z = BF16::to_float(((const u16*)a.gate_pre)[(int64_t)(q0 + tok) * a.gate_stride + head]);
    gsc = gsc / (1.0f + __expf(-z));
  }
  char* ob = smem_w + wave * 16 * RS;
#pragma unroll
  for (int db = 0; db < NDB; ++db) {         // 8-byte slot 4 db + g of row c, turned by the row within its 128 bytes
    if (!finishes(db)) continue;
    u16x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = BF16::from_float(acc[db][i] * gsc);
    *reinterpret_cast<u16x4*>(ob + c * RS + (((4 * db + g) ^ c) << 3)) = o;
  }
  if (two) __syncthreads();
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int j = 0; j < 16 * L / 64; ++j) {
    if (two && (j & 1) != group) continue;
    const int rl = (64 * j + lane) / L, ch = (64 * j + lane) % L, ro = row0 + rl;
    // slots 2 ch, 2 ch + 1 of row rl sit in chunk ch ^ (rl >> 1), in turned order when rl is odd
    u16x8 v = *reinterpret_cast<const u16x8*>(ob + rl * RS + 16 * (ch ^ (rl >> 1)));
    if (rl & 1) v = u16x8{v[4], v[5], v[6], v[7], v[0], v[1], v[2], v[3]};
    if (ro >= 0) *reinterpret_cast<u16x8*>((u16*)a.out + (int64_t)(q0 + ro / H) * a.out_token_stride + (int64_t)(ro % H) * a.out_head_stride + 8 * ch) = v;
  }
}

// The splits of a row merged: out = sum_s O_s 2^(m_s - M) / sum_s l_s 2^(m_s - M), times the head gate.  A row to R / 4 lanes (a power
// of two of them); one pass over the splits, four at a time, their loads all in flight together.
__global__ __launch_bounds__(256) void latent_attn_merge_kernel(hxm_latent_attn_args a, int tiles_per_seq, int lanes_log2) {
  const int R = a.kv_rank, H = a.n_heads, NS = a.n_splits, lanes = 1 << lanes_log2;
  const int64_t item = (((int64_t)blockIdx.x * 256 + threadIdx.x) >> lanes_log2);
  const int b = (int)(item / (tiles_per_seq * 16)), r = (int)(item % (tiles_per_seq * 16));
  if (b >= a.n_seq) return;
  const int q0 = a.q_cu[b];
  if (r >= (a.q_cu[b + 1] - q0) * H) return;
  const int t = q0 + r / H, h = r % H;
  const float* ml = a.ws_ml + 2 * (size_t)item * NS;
  float gate = 1.f;
  if (a.gate_pre) gate = 1.0f / (1.0f + __expf(-BF16::to_float(((const u16*)a.gate_pre)[(int64_t)t * a.gate_stride + h])));
  u16* og = (u16*)a.out + (int64_t)t * a.out_token_stride + (int64_t)h * a.out_head_stride;
  for (int c = 4 * ((int)threadIdx.x & (lanes - 1)); c < R; c += 4 * lanes) {
    const float* wo = a.ws_o + (size_t)item * NS * R + c;
    f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
    float M = HX_NEG_BIG, total = 0.f;
    for (int s0 = 0; s0 < NS; s0 += 4) {
      float mx[4], l[4];
      f32x4 v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int s = min(s0 + i, NS - 1);
        mx[i] = ml[2 * s];
        l[i] = ml[2 * s + 1];
        v[i] = *reinterpret_cast<const f32x4*>(wo + (size_t)s * R);
      }
      const float m_new = fmaxf(M, fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3])));
      const float keep = fast_exp2(M - m_new);
      total *= keep;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] *= keep;
      M = m_new;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float w = s0 + i < NS ? fast_exp2(mx[i] - M) : 0.f;
        total += w * l[i];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] += w * v[i][e];
      }
    }
    if (a.sinks) total += fast_exp2(a.sinks[h] * 1.4426950408889634f - M);      // the sink counts once, here
    const float gsc = gate / total;
    *reinterpret_cast<u16x4*>(og + c) = u16x4{BF16::from_float(o[0] * gsc), BF16::from_float(o[1] * gsc), BF16::from_float(o[2] * gsc), BF16::from_float(o[3] * gsc)};
  }
}

int prepare_lds(const void* kernel, size_t lds) {
  if (lds <= 48 * 1024) return HX_OK;
  const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e == hipSuccess) return HX_OK;
  hxm::last_hip_error() = (int)e;
  return HX_ERR_HIP;
}

// How the wide forms lay a launch out (the tile forms below keep the latents they do not take: widths or strides that are not whole
// 16-byte columns of 64, pages that are not whole 16-row groups).  rows32: waves of 32 rows (enough row tiles of 128 to fill the chip), else waves of 16 rows
// and the keys of a row tile dealt to `splits` workgroups where there are few of them.
struct WidePlan {
  bool fits, rows32;
  int splits, groups;
};
// keys that a portion looks at, at most
int key_reach(const hxm_latent_attn_args& a) {
  return a.window > 0 && a.window + a.max_q_len < a.max_kv_len ? a.window + a.max_q_len : a.max_kv_len;
}
WidePlan wide_plan(const hxm_latent_attn_args& a) {
  WidePlan p{false, false, 1, 1};
  if (a.kv_rank % 64 || a.block_size % 16 || a.out_token_stride % 8 || a.out_head_stride % 8 || !aligned16(a.out) || !aligned16(a.ws_o) ||
      a.cache_row_stride >= (1 << 26) || hxm::tile_form() != 1)
    return p;
  p.fits = true;
  const int64_t rows = (int64_t)a.max_q_len * a.n_heads;
  p.rows32 = a.kv_rank <= 192 && a.n_seq * ((rows + 127) / 128) >= 256;
  if (p.rows32) return p;
  if (hxm::latent_step_serves(a)) {
    p.splits = hxm::latent_step_splits(a);
    return p;
  }
  const int reach = key_reach(a);
  const int64_t tiles = a.n_seq * ((rows + 63) / 64);
  int64_t want = (512 + tiles - 1) / tiles;
  // (a split more shortens the walk over the keys and lengthens the writing and merging of what the splits hold, 8 bytes a row and
  //  column: their sum is least where the square of the splits is a multiple of keys / rows.  At 18, 36 and 72 times, 512 columns
  //  and 32 heads: 32 tokens of 301 - 1747 keys 36.4, 31.7, 30.5 us, under a window of 512 26, 25, 22.7; 16 tokens behind 4000
  //  keys 41, 37, 33; 16 portions of 4 behind 1000 keys 49, 35, 35.)
  while (want > 1 && want * want * a.n_seq * rows > (int64_t)72 * reach) --want;
  if (want > reach / 64) want = reach / 64;      // (two tiles of 32 keys a split at least)
  if (want > 64) want = 64;
  // One workgroup a compute unit leaves a SIMD one wave: two groups of waves share the keys, from seven tiles of them on (us, one group and two, 32 heads
  // on portions of 100 - 200 tokens: 50 keys of 256 columns 9.7 10.7, 195 of 320 17.5 17.4, 283 of 128 12.9 11.9, 450 of 256 25.2 21.9, 554 of 256 28.4 23.5) and in
  // the place of two splits, whose merge is a launch (one portion, 16 heads: 302 tokens of 320 columns 25.3 18.9, 922 of 128 29.3 22.2).  Three splits walk a third
  // of the keys each: two groups are faster only where the keys that a row sees, in the mean, are few: up to 500 in portions that bring a tenth of them and more
  // (eight heads on 948 tokens of 320 columns 32.9 25.7), 300 in shorter ones, where narrow rows are all that a split has to hand on (of 548 batches 5 %
  // in the mean, 26 slower by 2 - 8 %; behind the line, six portions of 28 tokens behind 1200, 256 columns, 27.7 35.7).  A compute unit takes one such
  // workgroup, so all of them have to be there at once: 320 portions of two tokens behind 520 keys, 256 columns, 24.7 33.1.  Up to 128 columns it takes two, and
  // from 400 keys on that is faster than one group each (16 heads on 198 and 845 tokens of 128 columns, 271 workgroups, 26.1 21.1; 250 keys 2 % slower).
  // More than 320 columns are more than a second group's sums leave registers for.
  const int64_t row_tiles = (int64_t)a.n_tokens * a.n_heads / 64 + a.n_seq;      // at most
  const bool narrow = a.kv_rank <= 320, at_once = row_tiles <= 256 || (a.kv_rank <= 128 && row_tiles <= 512 && reach >= 400);
  const int seen = reach - a.max_q_len / 2;      // in the mean
  const bool as_three = 10 * (int64_t)a.max_q_len >= reach ? seen <= 500 : a.kv_rank <= 192 && seen <= 300;
  if (narrow && at_once && (want < 2 ? reach >= 224 : want == 2 || (want == 3 && as_three))) {
    p.groups = 2;
  } else if (want > 1) {
    p.splits = (int)want;
  }
  return p;
}

template <int KK>
int launch_wide16(const hxm_latent_attn_args& a, int groups, hipStream_t s) {
  const int n_splits = a.n_splits > 1 ? a.n_splits : 1, tiles16 = (int)(((int64_t)a.max_q_len * a.n_heads + 15) / 16);
  const int64_t grid = (((int64_t)a.n_tokens * a.n_heads + 63) / 64 + a.n_seq) * n_splits;      // row tiles of all sequences, at most
  if (grid > 0x7fffffff) return HX_ERR_SHAPE;
  constexpr size_t images = 2 * 32 * 2 * 64 * KK;          // (of a group of waves)
  // (few rows: where the tile form would deal out the keys)
  const bool fine = n_splits > 1 || (int64_t)a.n_seq * tiles16 < kTileWaves;
  const bool two = KK <= 5 && fine && groups == 2;
  const size_t lds = two ? 2 * images + 4096 : images;
  auto kernel = fine ? latent_attn_wide16_kernel<KK, true, 1> : latent_attn_wide16_kernel<KK, false, 1>;
  if constexpr (KK <= 5) {
    if (two) kernel = latent_attn_wide16_kernel<KK, true, 2>;
  }
  if (const int rc = prepare_lds((const void*)kernel, lds)) return rc;
  kernel<<<dim3((unsigned)grid), dim3(two ? 512 : 256), lds, s>>>(a, tiles16);
  if (n_splits > 1) {
    int lanes_log2 = 4;                      // a row to R / 4 lanes, at most a power of two of them
    while ((8 << lanes_log2) <= a.kv_rank && lanes_log2 < 7) ++lanes_log2;
    const int64_t threads = ((int64_t)a.n_seq * tiles16 * 16) << lanes_log2;
    latent_attn_merge_kernel<<<dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s>>>(a, tiles16, lanes_log2);
  }
  return hxm::check_launch();
}

template <int KK>
int launch_wide(const hxm_latent_attn_args& a, const WidePlan& p, hipStream_t s) {
  if (a.n_splits > 1 && (a.n_splits > 64 || !a.ws_o || !a.ws_ml)) return HX_ERR_WORKSPACE;
  if constexpr (KK <= 3) {
    if (p.rows32) {
      const int64_t grid = ((int64_t)a.n_tokens * a.n_heads + 127) / 128 + a.n_seq;
      if (grid > 0x7fffffff) return HX_ERR_SHAPE;
      constexpr size_t lds = 2 * 64 * 2 * 64 * KK;
      if (const int rc = prepare_lds((const void*)latent_attn_wide_kernel<KK>, lds)) return rc;
      latent_attn_wide_kernel<KK><<<dim3((unsigned)grid), dim3(256), lds, s>>>(a);
      return hxm::check_launch();
    }
  }
  return hxm::latent_step_serves(a) ? hxm::launch_latent_step(a, s) : launch_wide16<KK>(a, p.groups, s);
}

// the splits of a (sequence, row tile) merged: out = sum_s O_s e^(m_s - M) / sum_s l_s e^(m_s - M), times the head gate
__global__ __launch_bounds__(256) void latent_attn_combine_kernel(hxm_latent_attn_args a, int tiles_per_seq) {
  const int64_t item = blockIdx.x;
  const int b = (int)(item / tiles_per_seq), tile = (int)(item % tiles_per_seq);
  const int H = a.n_heads, R = a.kv_rank, R16 = (R + 15) / 16 * 16, NS = a.n_splits;
  const int q0 = a.q_cu[b];
  const int n_rows = (a.q_cu[b + 1] - q0) * H;
  if (tile * 16 >= n_rows) return;
  __shared__ float wgt[16][65];      // [row][split] weight e^(m_s - M) / L (NS <= 64)
  if (threadIdx.x < 16) {
    const int row = threadIdx.x;
    const float* wml = a.ws_ml + (size_t)item * NS * 32;
    float M = -1.0e30f;
    for (int s = 0; s < NS; ++s) M = fmaxf(M, wml[s * 32 + 2 * row]);
    float L = 0.f;
    for (int s = 0; s < NS; ++s) L += wml[s * 32 + 2 * row + 1] * __expf(wml[s * 32 + 2 * row] - M);
    const int r = tile * 16 + row;
    if (a.sinks && r < n_rows) L += expf(a.sinks[r % H] - M);      // the sink counts once, here
    float gsc = L > 0.f ? 1.0f / L : 0.f;
    if (a.gate_pre && r < n_rows) {
      const float z = BF16::to_float(((const u16*)a.gate_pre)[(int64_t)(q0 + r / H) * a.gate_stride + r % H]);
      gsc = gsc / (1.0f + __expf(-z));
    }
    for (int s = 0; s < NS; ++s) wgt[row][s] = __expf(wml[s * 32 + 2 * row] - M) * gsc;
  }
  __syncthreads();
  const float* wo = a.ws_o + (size_t)item * NS * 16 * R16;
  for (int e = threadIdx.x; e < 16 * R; e += 256) {
    const int row = e / R, col = e % R;
    const int r = tile * 16 + row;
    if (r >= n_rows) continue;
    float v = 0.f;
    for (int s = 0; s < NS; ++s) v += wo[((size_t)s * 16 + row) * R16 + col] * wgt[row][s];
    ((u16*)a.out)[(int64_t)(q0 + r / H) * a.out_token_stride + (int64_t)(r % H) * a.out_head_stride + col] = BF16::from_float(v);
  }
}

// key splits for a launch: enough waves to fill the chip when there are few (sequence, row tile) items — decode steps
static int tile_splits(const hxm_latent_attn_args& a) {
  const int tiles_per_seq = (int)(((int64_t)a.max_q_len * a.n_heads + 15) / 16);
  const int64_t items = (int64_t)a.n_seq * tiles_per_seq;
  int reach = a.max_kv_len > 0 ? a.max_kv_len : 1;
  if (a.window > 0 && a.window + a.max_q_len < reach) reach = a.window + a.max_q_len;
  const int chunks = (reach + 31) / 32;
  int64_t want = (kTileWaves + items - 1) / items;
  if (want > chunks / 2) want = chunks / 2;          // at least two chunks a split
  if (want > 64) want = 64;
  return want < 2 ? 1 : (int)want;
}

template <int KK>
int launch_tile(const hxm_latent_attn_args& a, hipStream_t s) {
  const size_t per_wave = (size_t)32 * (2 * (KK * 32) + 32) + 16 * kPStride * 2;
  int waves = 4;
  while (waves > 1 && per_wave * waves > 64 * 1024) waves >>= 1;
  const int tiles_per_seq = (int)(((int64_t)a.max_q_len * a.n_heads + 15) / 16);
  const int n_splits = a.n_splits > 1 ? a.n_splits : 1;
  if (n_splits > 1 && (n_splits > 64 || !a.ws_o || !a.ws_ml)) return HX_ERR_WORKSPACE;
  // (measured: the group form wins where the tile form has no room for its second register set — latents of more than 256
  //  columns: 1136 -> 891 us at 512 columns — and loses below: 89 -> 140 us at 64 columns)
  if (KK > 8 && n_splits == 1 && tiles_per_seq >= 4 && hxm::tile_form() == 1) {
    const int groups_per_seq = (tiles_per_seq + 3) / 4;
    const size_t lds_g = (size_t)32 * (2 * (KK * 32) + 32) + 4 * 16 * kPStride * 2;
    latent_attn_group_kernel<KK><<<dim3((unsigned)((int64_t)a.n_seq * groups_per_seq)), dim3(256), lds_g, s>>>(a, groups_per_seq);
    return hxm::check_launch();
  }
  const int64_t items = (int64_t)a.n_seq * tiles_per_seq;
  const dim3 grid((unsigned)((items * n_splits + waves - 1) / waves));
  if constexpr (KK <= 8) latent_attn_tile_kernel<KK><<<grid, dim3(64 * waves), per_wave * waves, s>>>(a, tiles_per_seq, waves);
  else latent_attn_tile_wide_kernel<KK><<<grid, dim3(64 * waves), per_wave * waves, s>>>(a, tiles_per_seq, waves);
  if (n_splits > 1) latent_attn_combine_kernel<<<dim3((unsigned)items), dim3(256), 0, s>>>(a, tiles_per_seq);
  return hxm::check_launch();
}

}  // namespace

extern "C" int hxm_latent_norm_cache(const void* proj, int64_t proj_stride, int64_t q_off, int64_t q_rank, int64_t kv_off,
                                     int64_t kv_rank, const float* q_w, const float* kv_w, float eps, void* cq_out,
                                     const int32_t* slot_ids, void* cache, int64_t cache_block_stride,
                                     int64_t cache_row_stride, int32_t block_size, int64_t n_tokens, int dtype, void* stream) {
  if (n_tokens < 0 || q_rank < 1 || kv_rank < 1 || block_size < 1 || q_off < 0 || kv_off < 0) return HX_ERR_SHAPE;
  if (n_tokens == 0) return HX_OK;
  if (!proj || !q_w || !kv_w || !cq_out || !slot_ids || !cache) return HX_ERR_NULL;
  if (proj_stride < q_off + q_rank || proj_stride < kv_off + kv_rank || cache_row_stride < kv_rank) return HX_ERR_STRIDE;
  hipStream_t s = (hipStream_t)stream;
  const int64_t esz = dtype == HX_F32 ? 4 : 2;
  auto al = [&](const void* q, int64_t bytes) { return (reinterpret_cast<uintptr_t>(q) % bytes) == 0; };
  const int vec = (q_rank % 4 == 0 && kv_rank % 4 == 0 && q_off % 4 == 0 && kv_off % 4 == 0 && proj_stride % 4 == 0 &&
                   cache_row_stride % 4 == 0 && cache_block_stride % 4 == 0 && al(proj, 4 * esz) && al(cq_out, 4 * esz) &&
                   al(cache, 4 * esz) && al(q_w, 16) && al(kv_w, 16)) ? 1 : 0;
  switch (dtype) {
    case HX_F32:
      latent_norm_cache_kernel<F32><<<dim3((unsigned)((n_tokens + 3) / 4)), dim3(256), 0, s>>>(
          (const float*)proj, proj_stride, q_off, q_rank, kv_off, kv_rank, q_w, kv_w, eps, (float*)cq_out, slot_ids,
          (float*)cache, cache_block_stride, cache_row_stride, block_size, n_tokens, vec);
      break;
    case HX_BF16:
      latent_norm_cache_kernel<BF16><<<dim3((unsigned)((n_tokens + 3) / 4)), dim3(256), 0, s>>>(
          (const u16*)proj, proj_stride, q_off, q_rank, kv_off, kv_rank, q_w, kv_w, eps, (u16*)cq_out, slot_ids,
          (u16*)cache, cache_block_stride, cache_row_stride, block_size, n_tokens, vec);
      break;
    default: return HX_ERR_DTYPE;
  }
  return hxm::check_launch();
}

static bool tile_form_serves(const hxm_latent_attn_args& a) {
  const bool aligned = a.kv_rank % 8 == 0 && a.cache_row_stride % 8 == 0 && a.cache_block_stride % 8 == 0 &&
                       a.q_token_stride % 8 == 0 && a.q_head_stride % 8 == 0 && aligned16(a.cache) && aligned16(a.q);
  return a.dtype == HX_BF16 && aligned && a.kv_rank <= 512 && hxm::tile_form();
}

extern "C" int hxm_latent_attention_plan(const hxm_latent_attn_args* args, int32_t* n_splits, int64_t* ws_floats) {
  if (!args || !n_splits || !ws_floats) return HX_ERR_NULL;
  *n_splits = 1;
  *ws_floats = 0;
  if (args->n_tokens <= 0 || args->max_q_len < 1 || args->n_seq < 1 || !tile_form_serves(*args)) return HX_OK;
  const WidePlan p = wide_plan(*args);
  const int ns = p.fits ? p.splits : tile_splits(*args);
  if (ns > 1) {
    const int64_t tiles_per_seq = ((int64_t)args->max_q_len * args->n_heads + 15) / 16;
    const int64_t R16 = (args->kv_rank + 15) / 16 * 16;
    *n_splits = ns;
    *ws_floats = (int64_t)args->n_seq * tiles_per_seq * ns * 16 * (R16 + 2);
  }
  return HX_OK;
}

extern "C" int hxm_latent_attention_form(const hxm_latent_attn_args* args) {
  if (!args) return HX_ERR_NULL;
  if (args->max_q_len < 1 || !tile_form_serves(*args)) return HXM_LATENT_ROW;
  const WidePlan p = wide_plan(*args);
  return !p.fits ? HXM_LATENT_TILE : p.rows32 ? HXM_LATENT_WIDE32 : HXM_LATENT_WIDE16;
}

extern "C" int hxm_latent_attention(const hxm_latent_attn_args* args, void* stream) {
  if (!args) return HX_ERR_NULL;
  const hxm_latent_attn_args& a = *args;
  if (a.n_tokens < 0 || a.n_seq < 1 || a.n_heads < 1 || a.kv_rank < 1 || a.kv_rank > HXM_MAX_LATENT || a.block_size < 1)
    return HX_ERR_SHAPE;
  if (a.n_tokens == 0) return HX_OK;
  if (!a.out || !a.q || !a.cache || !a.tok_seq || !a.positions || !a.q_cu || !a.block_table || !a.cu_block_lens) return HX_ERR_NULL;
  if (a.cache_row_stride < a.kv_rank) return HX_ERR_STRIDE;
  hipStream_t s = (hipStream_t)stream;
  if (a.max_q_len < 1) return HX_ERR_SHAPE;
  if (tile_form_serves(a)) {
    const WidePlan p = wide_plan(a);
    if (p.fits) {
      switch (a.kv_rank / 64) {
        case 1: return launch_wide<1>(a, p, s);
        case 2: return launch_wide<2>(a, p, s);
        case 3: return launch_wide<3>(a, p, s);
        case 4: return launch_wide<4>(a, p, s);
        case 5: return launch_wide<5>(a, p, s);
        case 6: return launch_wide<6>(a, p, s);
        case 7: return launch_wide<7>(a, p, s);
        default: return launch_wide<8>(a, p, s);
      }
    }
    switch ((a.kv_rank + 31) / 32) {
      case 1: return launch_tile<1>(a, s);
      case 2: return launch_tile<2>(a, s);
      case 3: return launch_tile<3>(a, s);
      case 4: return launch_tile<4>(a, s);
      case 5: case 6: return launch_tile<6>(a, s);
      case 7: case 8: return launch_tile<8>(a, s);
      case 9: case 10: return launch_tile<10>(a, s);
      case 11: case 12: return launch_tile<12>(a, s);
      default: return launch_tile<16>(a, s);
    }
  }
  const int64_t items = (int64_t)a.n_tokens * a.n_heads;
  const dim3 grid((unsigned)((items + 3) / 4));
  const size_t lds = (size_t)4 * a.kv_rank * sizeof(float);
  switch (a.dtype) {
    case HX_F32: latent_attn_rows_kernel<F32><<<grid, dim3(256), lds, s>>>(a); break;
    case HX_BF16: latent_attn_rows_kernel<BF16><<<grid, dim3(256), lds, s>>>(a); break;
    default: return HX_ERR_DTYPE;
  }
  return hxm::check_launch();
}
