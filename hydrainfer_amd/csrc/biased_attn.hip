// biased_attn.hip — grouped-query attention over a paged key/value cache whose scores carry a linear distance bias,
// score(i, j) = q_i . k_j * scale - slope_h (i - j), under a causal, sliding-window or chunked mask (chunks counted from
// position 0 of the sequence).  Key and value rows may differ in size.  Scores, weights and sums are float.  Also the
// kernel in front of it: one RMS norm over a token's whole query projection and one over its whole key projection
// (all heads at once), keys and values straight into the cache.
#include <cfloat>
#include <algorithm>

#include "attn_common.h"
#include "mix_rows.h"
#include "../../include/hydra_mix.h"

namespace hxm {
int& last_hip_error();
int check_launch();
}  // namespace hxm

namespace {

using namespace hx;

// one workgroup per token.  vec: every offset, size, stride and pointer lets a lane move four elements at a time (and a
// head's key / value rows are multiples of four)
template <typename A>
__global__ __launch_bounds__(256) void qk_norm_cache_kernel(const typename A::storage* __restrict__ proj, int64_t proj_stride,
                                                            int64_t q_off, int64_t q_size, int64_t k_off, int64_t k_size,
                                                            int64_t v_off, int64_t v_size, const float* __restrict__ q_w,
                                                            const float* __restrict__ k_w, float eps,
                                                            typename A::storage* __restrict__ q_out,
                                                            const int32_t* __restrict__ slot_ids,
                                                            typename A::storage* __restrict__ key_cache,
                                                            typename A::storage* __restrict__ value_cache,
                                                            int64_t cache_row_stride, int64_t head_stride, int kv_heads, int vec) {
  __shared__ float part[8];
  const int64_t t = blockIdx.x;
  const typename A::storage* row = proj + t * proj_stride;
  const int step = vec ? 4 : 1;
  float ss[2] = {0.f, 0.f};      // sums of squares of the query and of the key projection, one pass
  if (q_w) {
    for (int64_t i = (int64_t)threadIdx.x * step; i < q_size; i += 256 * step) {
      if (vec) {
        const f32x4 v = Row4<A>::load(row + q_off + i);
        ss[0] += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
      } else {
        const float v = A::to_float(row[q_off + i]);
        ss[0] += v * v;
      }
    }
  }
  if (k_w) {
    for (int64_t i = (int64_t)threadIdx.x * step; i < k_size; i += 256 * step) {
      if (vec) {
        const f32x4 v = Row4<A>::load(row + k_off + i);
        ss[1] += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
      } else {
        const float v = A::to_float(row[k_off + i]);
        ss[1] += v * v;
      }
    }
  }
  if (q_w || k_w) block_sums<2>(ss, part);
  const float q_inv = 1.0f / sqrtf(ss[0] / (float)q_size + eps);
  for (int64_t i = (int64_t)threadIdx.x * step; i < q_size; i += 256 * step) {
    if (vec) {
      f32x4 v = Row4<A>::load(row + q_off + i);
      if (q_w) {
        const f32x4 w = *reinterpret_cast<const f32x4*>(q_w + i);
        v = f32x4{v[0] * q_inv * w[0], v[1] * q_inv * w[1], v[2] * q_inv * w[2], v[3] * q_inv * w[3]};
      }
      Row4<A>::store(q_out + t * q_size + i, v);
    } else {
      q_out[t * q_size + i] = q_w ? A::from_float(A::to_float(row[q_off + i]) * q_inv * q_w[i]) : row[q_off + i];
    }
  }
  if (k_size <= 0) return;
  const int64_t slot = slot_ids[t];
  if (slot < 0) return;
  const float k_inv = 1.0f / sqrtf(ss[1] / (float)k_size + eps);
  const int64_t kd = k_size / kv_heads, vd = v_size / kv_heads;
  typename A::storage* kr = key_cache + slot * cache_row_stride;
  typename A::storage* vr = value_cache + slot * cache_row_stride;
  for (int64_t i = (int64_t)threadIdx.x * step; i < k_size; i += 256 * step) {
    const int64_t at = (i / kd) * head_stride + i % kd;
    if (vec) {
      f32x4 v = Row4<A>::load(row + k_off + i);
      if (k_w) {
        const f32x4 w = *reinterpret_cast<const f32x4*>(k_w + i);
        v = f32x4{v[0] * k_inv * w[0], v[1] * k_inv * w[1], v[2] * k_inv * w[2], v[3] * k_inv * w[3]};
      }
      Row4<A>::store(kr + at, v);
    } else {
      kr[at] = k_w ? A::from_float(A::to_float(row[k_off + i]) * k_inv * k_w[i]) : row[k_off + i];
    }
  }
  for (int64_t i = (int64_t)threadIdx.x * step; i < v_size; i += 256 * step) {
    const int64_t at = (i / vd) * head_stride + i % vd;
    if (vec) Row4<A>::store(vr + at, Row4<A>::load(row + v_off + i));
    else vr[at] = row[v_off + i];
  }
}

// the wave's LDS writes so far are visible to all its lanes
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// a score under a soft cap: cap * tanh(s / cap); cap 0: the score itself
__device__ __forceinline__ float capped(float s, float cap) { return cap > 0.f ? cap * tanhf(s / cap) : s; }

// tanh(y) as exact near 0 as elsewhere, for y within kCapNear: an odd polynomial (its even part fitted to equal relative error, 5e-9); any y:
// beyond it 1 - 2 / (1 + e^(2 |y|)) with y's sign.  (That form near 0 is off by a share of the cap and not of the score.)
constexpr float kCapNear = 0.625f;
__device__ __forceinline__ float tanh_near(float y) {
  const float t = y * y;
  const float p = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(__builtin_fmaf(-0.00570500642f, t, 0.0206391029f), t, -0.0537397191f), t, 0.133314416f), t, -0.333332807f);
  return __builtin_fmaf(y * t, p, y);
}
__device__ __forceinline__ float tanh_any(float y) {
  const float far = __builtin_fmaf(-2.f, __builtin_amdgcn_rcpf(1.f + fast_exp2(fabsf(y) * 2.8853900817779268f)), 1.f);
  return fabsf(y) < kCapNear ? tanh_near(y) : copysignf(far, y);
}
// N scores times unit under a cap, times cap2.  Scores far below the cap are the rule: nothing but the polynomial then (4 portions of 797
// - 1151 tokens, 32 / 8 heads of 128, window of 512: no cap 56 us, a cap of 30 68 us, a cap of 1, which takes both ways, 87).
template <int N, typename S>
__device__ __forceinline__ void cap_scores(S& s, float unit, float cap2) {
  float top = 0.f;
#pragma unroll
  for (int e = 0; e < N; ++e) {
    s[e] *= unit;
    top = fmaxf(top, fabsf(s[e]));
  }
  if (__builtin_amdgcn_ballot_w64(top >= kCapNear)) {
#pragma unroll
    for (int e = 0; e < N; ++e) s[e] = tanh_any(s[e]) * cap2;
  } else {
#pragma unroll
    for (int e = 0; e < N; ++e) s[e] = tanh_near(s[e]) * cap2;
  }
}

// D[32 x 32] += A[32 x 16] B[16 x 32]; lane (c = l % 32, h = l / 32): A[c][8 h + j], B[8 h + j][c], D[(e & 3) + 8 (e / 4) + 4 h][c]
__device__ __forceinline__ f32x16 mma32(u16x8 a, u16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// the first key a query at position i sees
__device__ __forceinline__ int first_visible(int i, int kind, int size) {
  if (kind == HXM_MASK_WINDOW) return i - size + 1 > 0 ? i - size + 1 : 0;
  if (kind == HXM_MASK_CHUNK) return i / size * size;
  return 0;
}

// ---------------------------------------------------------------------------------------------------------------
// Row form: one wave per (token, head), four a workgroup, no barriers.  Keys go by in groups of 64: lane l scores key
// lo + l (its row of the cache against the query in LDS), the group's maximum and sum are wave reductions, then the lanes
// turn to the value's columns (lane l owns columns l, l + 64, ...) and add the 64 rows, each weighted by its lane's p.
// ---------------------------------------------------------------------------------------------------------------
constexpr int kMaxVCols = 8;      // value columns per lane: vdim <= 512
template <typename A>
__global__ __launch_bounds__(256) void biased_attn_rows_kernel(hxm_biased_attn_args a) {
  extern __shared__ float lds[];
  typedef typename A::storage T;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t item = (int64_t)blockIdx.x * 4 + wave;
  if (item >= (int64_t)a.n_tokens * a.n_heads) return;
  const int t = (int)(item / a.n_heads), h = (int)(item - (int64_t)t * a.n_heads);
  const int D = a.dim, V = a.vdim, BS = a.block_size;
  float* qs = lds + wave * (D + 64);       // the query, then the group's weights
  float* ps = qs + D;
  const T* q = (const T*)a.q + ((int64_t)t * a.n_heads + h) * D;
  const float qscale = a.head_scale ? a.scale * a.head_scale[h] : a.scale;
  for (int d = lane; d < D; d += 64) qs[d] = A::to_float(q[d]) * qscale;
  wave_lds_sync();
  const int seq = a.tok_seq[t], i = a.positions[t];
  const int32_t* table = a.block_table + a.cu_block_lens[seq];
  const int g = h / (a.n_heads / a.kv_heads);
  const T* kc = (const T*)a.key_cache + (int64_t)g * a.head_stride;
  const T* vc = (const T*)a.value_cache + (int64_t)g * a.head_stride;
  const float slope = a.slopes ? a.slopes[h] : 0.f;
  const int lo = first_visible(i, a.mask_kind, a.mask_size);
  float m = -FLT_MAX, l = 0.f;
  float acc[kMaxVCols];
#pragma unroll
  for (int c = 0; c < kMaxVCols; ++c) acc[c] = 0.f;
  for (int j0 = lo; j0 <= i; j0 += 64) {
    const int j = j0 + lane;
    float s = -FLT_MAX;
    if (j <= i) {
      const T* kr = kc + (int64_t)table[j / BS] * a.cache_block_stride + (int64_t)(j % BS) * a.cache_row_stride;
      float dot = 0.f;
      for (int d = 0; d < D; ++d) dot += qs[d] * A::to_float(kr[d]);
      if (a.softcap > 0.f) dot = a.softcap * tanhf(dot / a.softcap);
      s = dot - slope * (float)(i - j);
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float p = j <= i ? expf(s - m_new) : 0.f;
    const float corr = expf(m - m_new);
    l = l * corr + wave_sum(p);
    m = m_new;
    wave_lds_sync();
    ps[lane] = p;
    wave_lds_sync();
#pragma unroll
    for (int c = 0; c < kMaxVCols; ++c) acc[c] *= corr;
    const int n = i - j0 + 1 < 64 ? i - j0 + 1 : 64;
    for (int jj = 0; jj < n; ++jj) {
      const int jk = j0 + jj;
      const T* vr = vc + (int64_t)table[jk / BS] * a.cache_block_stride + (int64_t)(jk % BS) * a.cache_row_stride;
      const float pj = ps[jj];
#pragma unroll
      for (int c = 0; c < kMaxVCols; ++c) {
        const int col = lane + 64 * c;
        if (col < V) acc[c] += pj * A::to_float(vr[col]);
      }
    }
  }
  T* o = (T*)a.out + ((int64_t)t * a.n_heads + h) * V;
  if (a.sinks) l += expf(a.sinks[h] - m);      // the sink: one more term of the denominator, without a value
  const float inv = 1.0f / l;
#pragma unroll
  for (int c = 0; c < kMaxVCols; ++c) {
    const int col = lane + 64 * c;
    if (col < V) o[col] = A::from_float(acc[c] * inv);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Tile form (bfloat16): one wave per 16 rows, a row being a (token, query head) pair of ONE sequence's portion and ONE
// key/value head, the group's query heads fastest — the heads of a decoded token that share a key head, or a few tokens
// times those heads.  All rows of a tile read the same keys, which go by in chunks of 32: S = Q K^T and O += P V are
// 16x16x32 MFMAs.  Key rows come straight from the paged cache into the B operands of S (a lane's 16 bytes are 8
// consecutive columns of one key's row); value rows are written to the wave's LDS as they come (row-major image of the
// chunk) and return through the transposing LDS read as B operands of the second product; P goes through LDS from the
// accumulator layout to the A layout.  Bias and mask are applied to the float scores, row by row.  With n_splits > 1 the
// key range of a tile is dealt to several waves whose partial results a second kernel merges.  No workgroup barriers.
// ---------------------------------------------------------------------------------------------------------------
constexpr int kPStride = 36;       // u16 per row of P in LDS: 32 slots + 4

template <int KK>                  // ceil(max(dim, vdim) / 32): 1, 2, 4, 8
__global__ __launch_bounds__(256) void biased_attn_tile_kernel(hxm_biased_attn_args a, int tiles_per_seq, int waves_per_block) {
  extern __shared__ float lds[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (wave >= waves_per_block) return;
  const int n_splits = a.n_splits > 1 ? a.n_splits : 1;
  const int G = a.kv_heads, R = a.n_heads / a.kv_heads, D = a.dim, V = a.vdim;
  const int64_t witem = (int64_t)blockIdx.x * waves_per_block + wave;      // (sequence, kv head, row tile, key split), splits fastest
  if (witem >= (int64_t)a.n_seq * G * tiles_per_seq * n_splits) return;
  const int64_t item = witem / n_splits;
  const int split = (int)(witem % n_splits);
  const int tile = (int)(item % tiles_per_seq);
  const int kvh = (int)((item / tiles_per_seq) % G);
  const int b = (int)(item / ((int64_t)tiles_per_seq * G));
  const int q0 = a.q_cu[b];
  const int n_rows = (a.q_cu[b + 1] - q0) * R;
  if (tile * 16 >= n_rows) return;
  const int g = lane >> 4, c = lane & 15;
  const int RS = 2 * (KK * 32) + 32;      // bytes per row of the value image (a key's columns, padded)
  char* img = reinterpret_cast<char*>(lds) + (size_t)wave * (32 * RS + 16 * kPStride * 2);
  u16* pl = reinterpret_cast<u16*>(img + 32 * RS);
  const u16* kc = (const u16*)a.key_cache + (int64_t)kvh * a.head_stride;
  const u16* vc = (const u16*)a.value_cache + (int64_t)kvh * a.head_stride;
  const int32_t* table = a.block_table + a.cu_block_lens[b];
  const u16x8 zero8 = u16x8{0, 0, 0, 0, 0, 0, 0, 0};

  // the queries: lane (g, c) holds row c, columns 32 kk + 8 g .. + 7
  const int last_row = min(tile * 16 + 15, n_rows - 1);
  u16x8 qf[KK];
  {
    const int r = min(tile * 16 + c, n_rows - 1);
    const u16* qg = (const u16*)a.q + ((int64_t)(q0 + r / R) * a.n_heads + kvh * R + r % R) * D;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const int col = 32 * kk + 8 * g;
      qf[kk] = col < D ? *reinterpret_cast<const u16x8*>(qg + col) : zero8;
    }
  }
  // the rows this lane holds of S and O: 4 g + i
  int pos[4], lo[4];
  float slope[4], hsc[4], snk[4];      // per row: distance slope, score scale (scale * head_scale), sink term's logit
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = tile * 16 + 4 * g + i;
    hsc[i] = a.scale;
    snk[i] = -INFINITY;
    if (r < n_rows) {
      const int h = kvh * R + r % R;
      pos[i] = a.positions[q0 + r / R];
      lo[i] = first_visible(pos[i], a.mask_kind, a.mask_size);
      slope[i] = a.slopes ? a.slopes[h] : 0.f;
      if (a.head_scale) hsc[i] = a.scale * a.head_scale[h];
      if (a.sinks) snk[i] = a.sinks[h];
    } else {
      pos[i] = -1;      // sees nothing
      lo[i] = 0;
      slope[i] = 0.f;
    }
  }
  // the keys any row of the tile sees
  int k_min, k_max;
  {
    const int r = min(tile * 16 + c, last_row);
    const int pr = a.positions[q0 + r / R];
    k_max = pr;
    k_min = first_visible(pr, a.mask_kind, a.mask_size);
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
  int k_begin = k_min, k_end = k_max;
  if (n_splits > 1) {
    const int chunks = (k_max - k_min + 32) / 32;
    const int per = (chunks + n_splits - 1) / n_splits;
    k_begin = k_min + split * per * 32;
    k_end = min(k_max, k_begin + per * 32 - 1);
  }
  const int bs = a.block_size;
  const int bshift = (bs & (bs - 1)) == 0 ? __ffs(bs) - 1 : -1;
  // a chunk's key or value rows, this lane's part: key 16 s + c, columns 32 kk + 8 g .. + 7
  auto fetch = [&](int key0, const u16* base, int width, u16x8 (&f)[2][KK]) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int key = min(key0 + 16 * s + c, k_max);        // (a key past the last one repeats it; masked below)
      const int page = bshift >= 0 ? key >> bshift : key / bs;
      const int64_t off = (int64_t)table[page] * a.cache_block_stride + (int64_t)(key - page * bs) * a.cache_row_stride;
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        const int col = 32 * kk + 8 * g;
        f[s][kk] = col < width ? *reinterpret_cast<const u16x8*>(base + off + col) : zero8;
      }
    }
  };
  // One register set each for keys and values: a chunk's values are asked for before its scores are multiplied, and the
  // next chunk's keys as soon as the scores are done — both loads are in flight behind the softmax and the products.
  u16x8 kf[2][KK], vf[2][KK];
  if (k_begin <= k_end) fetch(k_begin, kc, D, kf);
  for (int key0 = k_begin; key0 <= k_end; key0 += 32) {
    fetch(key0, vc, V, vf);
    f32x4 sc[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      sc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) sc[s] = Mfma<BF16>::mma(qf[kk], kf[s][kk], sc[s]);
    }
    if (key0 + 32 <= k_end) fetch(key0 + 32, kc, D, kf);
    // softmax of the rows 4 g + i over this chunk (sc[s][i] is key key0 + 16 s + c)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float p[2];
      float mx = -INFINITY;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int key = key0 + 16 * s + c;
        const bool seen = key >= lo[i] && key <= pos[i];
        p[s] = seen ? capped(sc[s][i] * hsc[i], a.softcap) - slope[i] * (float)(pos[i] - key) : -INFINITY;
        mx = fmaxf(mx, p[s]);
      }
      mx = row16_max(mx);      // (the sixteen lanes that hold the row's scores: one DPP row)
      const float m_new = fmaxf(m[i], mx);
      const float corr = __expf(m[i] - m_new);
      p[0] = __expf(p[0] - m_new);       // exp(-inf) = 0 for a key the row does not see
      p[1] = __expf(p[1] - m_new);
      float ps = p[0] + p[1];
      ps = row16_sum(ps);
      l[i] = l[i] * corr + ps;
      m[i] = m_new;
#pragma unroll
      for (int n = 0; n < KK * 2; ++n) acc[n][i] *= corr;
      // key 16 s + c sits in slot 8 (c / 4) + c % 4 + 4 s of its row: the order the transposing read delivers the keys in
      pl[(4 * g + i) * kPStride + 8 * (c >> 2) + (c & 3)] = BF16::from_float(p[0]);
      pl[(4 * g + i) * kPStride + 8 * (c >> 2) + (c & 3) + 4] = BF16::from_float(p[1]);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) *reinterpret_cast<u16x8*>(img + (16 * s + c) * RS + (32 * kk + 8 * g) * 2) = vf[s][kk];
    wave_lds_sync();
    // O += P V: A = P[row c][slots 8 g ..], B = the image's column 16 n + c at the keys of those slots
    u16x8 pf;
    {
      const u16x4 x0 = *reinterpret_cast<const u16x4*>(pl + c * kPStride + 8 * g);
      const u16x4 x1 = *reinterpret_cast<const u16x4*>(pl + c * kPStride + 8 * g + 4);
      pf = u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
    }
    const char* vrd = img + (4 * g + (c >> 2)) * RS + (c & 3) * 8;
#pragma unroll
    for (int n = 0; n < KK * 2; ++n) {
      const u16x4 x0 = lds_tr_read(vrd + n * 32);
      const u16x4 x1 = lds_tr_read(vrd + 16 * RS + n * 32);
      const u16x8 vv = u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
      acc[n] = Mfma<BF16>::mma(pf, vv, acc[n]);
    }
    wave_lds_sync();      // the reads are done before the next chunk is written
  }
  const int V16 = (V + 15) / 16 * 16;
  if (n_splits > 1) {
    // unnormalised partial result of this split: ws_o [item][split][16 rows][V16], ws_ml [item][split][16 rows][m, l]
    float* wo = a.ws_o + ((size_t)witem * 16) * V16;
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
        if (col < V16) wo[(size_t)row * V16 + col] = acc[n][i];
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = tile * 16 + 4 * g + i;
    if (r >= n_rows) continue;
    const float inv = 1.0f / (l[i] + expf(snk[i] - m[i]));      // (no sink: exp(-inf) = 0)
    u16* og = (u16*)a.out + ((int64_t)(q0 + r / R) * a.n_heads + kvh * R + r % R) * V;
#pragma unroll
    for (int n = 0; n < KK * 2; ++n) {
      const int col = 16 * n + c;
      if (col < V) og[col] = BF16::from_float(acc[n][i] * inv);
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Group form (bfloat16, portions of prompts, head sizes up to 128): a workgroup of four waves takes four consecutive row
// tiles (64 rows) of ONE (sequence, key head) and ONE image of every 32-key chunk.  The tile form is bound by its loads —
// sixteen 16-byte load instructions per chunk and wave, each touching sixteen half cache lines; here the workgroup brings
// a chunk's key and value rows once, in whole rows (two to four loads a thread), into one of two LDS images, and all four
// waves read the B operands of both products from there (16-byte reads for S, transposing reads for O).  The next chunk
// is on its way into registers while this one is multiplied and goes to the other image afterwards: one workgroup barrier
// a chunk, one that orders LDS only.  A wave skips the chunks none of its rows sees.
// ---------------------------------------------------------------------------------------------------------------
template <int KK>                  // ceil(max(dim, vdim) / 32): 1, 2, 4
__global__ __launch_bounds__(256) void biased_attn_group_kernel(hxm_biased_attn_args a, int groups_per_seq) {
  extern __shared__ float lds[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int G = a.kv_heads, R = a.n_heads / a.kv_heads, D = a.dim, V = a.vdim;
  const int64_t item = blockIdx.x;                                   // (sequence, kv head, group of four row tiles)
  const int group = (int)(item % groups_per_seq);
  const int kvh = (int)((item / groups_per_seq) % G);
  const int b = (int)(item / ((int64_t)groups_per_seq * G));
  const int q0 = a.q_cu[b];
  const int n_rows = (a.q_cu[b + 1] - q0) * R;
  if (group * 64 >= n_rows) return;                                  // (the whole workgroup: no barrier is left waiting)
  const int tile = group * 4 + wave;
  const bool live = tile * 16 < n_rows;                              // a wave past the portion's rows only helps to load
  const int g = lane >> 4, c = lane & 15;
  constexpr int RS = 2 * (KK * 32) + 32;                             // bytes per row of an image (a key's columns, padded)
  constexpr int PR = KK * 4;                                         // 16-byte pieces per row
  constexpr int NP = (32 * PR + 255) / 256;                          // pieces of a chunk's keys (or values) a thread brings
  char* base = reinterpret_cast<char*>(lds);
  char* img_k[2] = {base, base + 32 * RS};
  char* img_v[2] = {base + 64 * RS, base + 96 * RS};
  u16* pl = reinterpret_cast<u16*>(base + 128 * RS) + wave * (16 * kPStride);
  const u16* kc = (const u16*)a.key_cache + (int64_t)kvh * a.head_stride;
  const u16* vc = (const u16*)a.value_cache + (int64_t)kvh * a.head_stride;
  const int32_t* table = a.block_table + a.cu_block_lens[b];
  const u16x8 zero8 = u16x8{0, 0, 0, 0, 0, 0, 0, 0};

  u16x8 qf[KK];
  {
    const int r = min(tile * 16 + c, n_rows - 1);
    const u16* qg = (const u16*)a.q + ((int64_t)(q0 + r / R) * a.n_heads + kvh * R + r % R) * D;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const int col = 32 * kk + 8 * g;
      qf[kk] = col < D ? *reinterpret_cast<const u16x8*>(qg + col) : zero8;
    }
  }
  int pos[4], lo[4];
  float slope[4], hsc[4], snk[4];      // per row: distance slope, score scale (scale * head_scale), sink term's logit
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = tile * 16 + 4 * g + i;
    hsc[i] = a.scale;
    snk[i] = -INFINITY;
    if (r < n_rows) {
      const int h = kvh * R + r % R;
      pos[i] = a.positions[q0 + r / R];
      lo[i] = first_visible(pos[i], a.mask_kind, a.mask_size);
      slope[i] = a.slopes ? a.slopes[h] : 0.f;
      if (a.head_scale) hsc[i] = a.scale * a.head_scale[h];
      if (a.sinks) snk[i] = a.sinks[h];
    } else {
      pos[i] = -1;      // sees nothing
      lo[i] = 0;
      slope[i] = 0.f;
    }
  }
  // rows of a portion are in the order of their positions: the group's first row sees the earliest key, its last the latest
  const int k_begin = first_visible(a.positions[q0 + (group * 64) / R], a.mask_kind, a.mask_size);
  const int k_end = a.positions[q0 + min(group * 64 + 63, n_rows - 1) / R];
  int w_min = 0x7fffffff, w_max = -1;      // the keys this wave's rows see
  if (live) {
    w_min = first_visible(a.positions[q0 + (tile * 16) / R], a.mask_kind, a.mask_size);
    w_max = a.positions[q0 + min(tile * 16 + 15, n_rows - 1) / R];
  }
  float m[4], l[4];
  f32x4 acc[KK * 2];
#pragma unroll
  for (int i = 0; i < 4; ++i) { m[i] = -1.0e30f; l[i] = 0.f; }
#pragma unroll
  for (int n = 0; n < KK * 2; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int bs = a.block_size;
  const int bshift = (bs & (bs - 1)) == 0 ? __ffs(bs) - 1 : -1;
  // piece p of a chunk: row p / PR (a key), columns 8 (p % PR) .. + 7
  u16x8 kr[NP], vr[NP];
  auto fetch = [&](int key0) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      const int p = threadIdx.x + 256 * n;
      kr[n] = zero8;
      vr[n] = zero8;
      if (p < 32 * PR) {
        const int key = min(key0 + p / PR, k_end), col = (p % PR) * 8;      // (a key past the last one repeats it; masked below)
        const int page = bshift >= 0 ? key >> bshift : key / bs;
        const int64_t off = (int64_t)table[page] * a.cache_block_stride + (int64_t)(key - page * bs) * a.cache_row_stride + col;
        if (col < D) kr[n] = *reinterpret_cast<const u16x8*>(kc + off);
        if (col < V) vr[n] = *reinterpret_cast<const u16x8*>(vc + off);
      }
    }
  };
  auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      const int p = threadIdx.x + 256 * n;
      if (p < 32 * PR) {
        const int at = (p / PR) * RS + (p % PR) * 16;
        *reinterpret_cast<u16x8*>(img_k[buf] + at) = kr[n];
        *reinterpret_cast<u16x8*>(img_v[buf] + at) = vr[n];
      }
    }
  };
  fetch(k_begin);
  store(0);
  lds_barrier();
  int buf = 0;
  for (int key0 = k_begin; key0 <= k_end; key0 += 32, buf ^= 1) {
    const bool more = key0 + 32 <= k_end;
    if (more) fetch(key0 + 32);
    if (key0 <= w_max && key0 + 31 >= w_min) {
      f32x4 sc[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        sc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          const u16x8 kf = *reinterpret_cast<const u16x8*>(img_k[buf] + (16 * s + c) * RS + (32 * kk + 8 * g) * 2);
          sc[s] = Mfma<BF16>::mma(qf[kk], kf, sc[s]);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float p[2];
        float mx = -INFINITY;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int key = key0 + 16 * s + c;
          const bool seen = key >= lo[i] && key <= pos[i];
          p[s] = seen ? capped(sc[s][i] * hsc[i], a.softcap) - slope[i] * (float)(pos[i] - key) : -INFINITY;
          mx = fmaxf(mx, p[s]);
        }
        mx = row16_max(mx);
        const float m_new = fmaxf(m[i], mx);
        const float corr = __expf(m[i] - m_new);
        p[0] = __expf(p[0] - m_new);
        p[1] = __expf(p[1] - m_new);
        float ps = p[0] + p[1];
        ps = row16_sum(ps);
        l[i] = l[i] * corr + ps;
        m[i] = m_new;
#pragma unroll
        for (int n = 0; n < KK * 2; ++n) acc[n][i] *= corr;
        pl[(4 * g + i) * kPStride + 8 * (c >> 2) + (c & 3)] = BF16::from_float(p[0]);
        pl[(4 * g + i) * kPStride + 8 * (c >> 2) + (c & 3) + 4] = BF16::from_float(p[1]);
      }
      wave_lds_sync();
      u16x8 pf;
      {
        const u16x4 x0 = *reinterpret_cast<const u16x4*>(pl + c * kPStride + 8 * g);
        const u16x4 x1 = *reinterpret_cast<const u16x4*>(pl + c * kPStride + 8 * g + 4);
        pf = u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
      }
      const char* vrd = img_v[buf] + (4 * g + (c >> 2)) * RS + (c & 3) * 8;
#pragma unroll
      for (int n = 0; n < KK * 2; ++n) {
        const u16x4 x0 = lds_tr_read(vrd + n * 32);
        const u16x4 x1 = lds_tr_read(vrd + 16 * RS + n * 32);
        const u16x8 vv = u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
        acc[n] = Mfma<BF16>::mma(pf, vv, acc[n]);
      }
      wave_lds_sync();      // this wave's reads of P are done before it writes the next chunk's
    }
    if (more) store(buf ^ 1);      // (the other image: every wave finished with it before the last barrier)
    lds_barrier();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = tile * 16 + 4 * g + i;
    if (r >= n_rows) continue;
    const float inv = 1.0f / (l[i] + expf(snk[i] - m[i]));      // (no sink: exp(-inf) = 0)
    u16* og = (u16*)a.out + ((int64_t)(q0 + r / R) * a.n_heads + kvh * R + r % R) * V;
#pragma unroll
    for (int n = 0; n < KK * 2; ++n) {
      const int col = 16 * n + c;
      if (col < V) og[col] = BF16::from_float(acc[n][i] * inv);
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Wide form (bfloat16, portions of prompts, key and value heads of 64 or 128, pages of whole 16-row groups): a workgroup of four
// waves takes 128 rows, 32 a wave, of ONE (sequence, key head) and goes over the keys in tiles of 64.  The group form is bound by
// LDS reads (a 16-byte read feeds one 16 x 16 x 32 product) and by the vector work of its softmax; here
//   * the products are 32 x 32 x 16 and swapped, S^T = K Q^T and O^T += V^T P^T: a row of the softmax is one lane (its mask,
//     slope, temperature are scalars of the lane, its maximum and sum one exchange with lane + 32), and P goes into the second
//     product from the registers it was made in;
//   * a tile's key and value rows go straight from the paged cache to LDS (1 KiB an instruction, whole rows), the next tile's
//     while this one is worked on: two images, one barrier a tile.  Rows cannot be padded this way; their 16-byte chunks are
//     swizzled by the lane that asks for them (keys: chunk ^ row, values: 64-byte quarter ^ row);
//   * a row's weights refer to its largest score so far, 32 keys at a time, and their sum is that of the floats.  That costs a pass over the
//     accumulators for nearly every half tile; left up to 2^8 behind, it took 5 us less and results were off by 3 % more, as the largest
//     weights were rounded to bfloat16 instead of being 1.  (64 keys at a time behind a workgroup's first two tiles, and sums of the rounded
//     weights: 1 us less, and off by more where all of a row's keys lie in such tiles, as behind the edge of a chunk.)
//   * where workgroups are few, two groups of four waves take every other tile of keys each, with images of their own, and add up what they have at
//     the end: each hands the other half of its columns through LDS, scaled like the splits of a row (a wave alone on its SIMD goes from products
//     to softmax to products, 2 - 3 us a tile).
// The order of the row tiles: the XCDs (workgroups are dealt round robin) take key heads of their own where there are enough of
// them, and of every sequence the tiles with the most keys come first.
// Measured, 4 portions of 797 - 1151 tokens, 32 heads of 128 on 8 key heads, sinks: 221 us in the group form, 55 us
// here (580 TFLOP/s of the pairs that a mask leaves); window of 512 and soft cap 223 and 68 us; chunks of 512 and slopes 163 and
// 50 us.  Down to 64 rows of a key head it is the faster one (16 tokens behind 500 keys: 30 and 21 us).
// ---------------------------------------------------------------------------------------------------------------
template <int D, int V, bool MODS, bool FINE, int KG>      // MODS: slopes or a soft cap; FINE: every 32 keys' weights refer to their own largest score; KG: groups of four waves
__global__ __launch_bounds__(256 * KG, 2) void biased_attn_wide_kernel(hxm_biased_attn_args a, int tile_slots) {
  constexpr int KT = 64, TQ = 128, KS = D / 16, NDB = V / 32;
  constexpr int RSK = 2 * D, RSV = 2 * V, LK = D / 8, LV = V / 8;        // bytes and 16-byte chunks of a row
  constexpr int KTILE = KT * RSK, IMG = KTILE + KT * RSV;
  extern __shared__ __attribute__((aligned(16))) char smem_w[];        // [KG][2][K tile | V tile]
  auto kswz = [](int row) { return LK == 16 ? (row & 15) : ((row >> 1) & 7); };
  auto vswz = [](int row) { return LV == 16 ? ((row & 3) << 2) : (((row >> 1) & 1) << 2); };
  typedef __attribute__((address_space(4))) const int32_t c_i32;       // (uniform indices: through the scalar cache)
  c_i32* q_cu = (c_i32*)a.q_cu;
  const int G = a.kv_heads, R = a.n_heads / a.kv_heads;

  // workgroup -> (sequence, row tile, key head): within a sequence the last tiles, which see the most keys, first
  int kvh, slot;
  {
    const int wg = blockIdx.x, total = tile_slots * G;
    if (G % 8 == 0) {                        // XCD x: key heads x G / 8 ..
      const int hp = G / 8, i = wg >> 3;
      kvh = (wg & 7) * hp + i % hp;
      slot = i / hp;
    } else {
      kvh = wg / tile_slots;
      slot = wg - kvh * tile_slots;
    }
    if (wg >= total) return;
  }
  int b, tile, q0, n_rows;
  if (!find_row_tile<TQ>(q_cu, a.n_seq, R, slot, b, tile, q0, n_rows)) return;      // spare slot (the grid is an upper bound)
  const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3), lane = threadIdx.x & 63;
  const int group = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;      // takes every KG-th tile of keys
  const int c = lane & 31, hi = lane >> 5;
  // row tiles end with the portion: a partial one is the first, with the fewest keys.  Rows below 0 do not exist.
  const int row0_wg = n_rows - ((n_rows + TQ - 1) / TQ - tile) * TQ, row0 = row0_wg + 32 * wave;
  const int r = max(row0 + c, 0), tok = r / R, head = kvh * R + r % R;
  const int pos = a.positions[q0 + tok];
  const int lo = first_visible(pos, a.mask_kind, a.mask_size);
  // what the rows of the wave see, and any row of the workgroup (every wave looks at all of them: no order of the positions is assumed)
  const int wpos0 = wave_min_int(pos), wpos1 = wave_max_int(pos), wlo0 = wave_min_int(lo), wlo1 = wave_max_int(lo);
  int k_first, k_last;
  {
    const int p0 = a.positions[q0 + max(row0_wg + lane, 0) / R], p1 = a.positions[q0 + max(row0_wg + 64 + lane, 0) / R];
    k_first = wave_min_int(min(first_visible(p0, a.mask_kind, a.mask_size), first_visible(p1, a.mask_kind, a.mask_size)));
    k_last = wave_max_int(max(p0, p1));
  }
  const bool live = row0 + 31 >= 0;
  const int t_first = k_first / KT, t_last = k_last < 0 ? t_first - 1 : k_last / KT;      // (positions below 0 see nothing)

  const u16* kc = (const u16*)a.key_cache + (int64_t)kvh * a.head_stride;
  const u16* vc = (const u16*)a.value_cache + (int64_t)kvh * a.head_stride;
  c_i32* table = (c_i32*)(a.block_table + ((c_i32*)a.cu_block_lens)[b]);
  const int bs = a.block_size, bshift = (bs & (bs - 1)) == 0 ? __ffs(bs) - 1 : -1;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem_w + (uint32_t)(group * 2 * IMG);
  // Wave w brings keys 16 w .. of a tile (one page): RPK / RPV rows an instruction, LK / LV lanes a row.  What lies in front of the
  // first key that some row sees, or behind the last, is not touched (its page may be gone): rows there repeat that key, masked.
  constexpr int RPK = 64 / LK, RPV = 64 / LV;
  const int rk = lane / LK, ck = lane % LK, rv = lane / LV, cv = lane % LV;
  uint32_t ko[16 / RPK], vo[16 / RPV];       // a lane's part of a group of sixteen whole rows, in bytes
#pragma unroll
  for (int j = 0; j < 16 / RPK; ++j) ko[j] = (uint32_t)(2 * ((RPK * j + rk) * (uint32_t)a.cache_row_stride + 8 * (ck ^ kswz(RPK * j + rk))));
#pragma unroll
  for (int j = 0; j < 16 / RPV; ++j) vo[j] = (uint32_t)(2 * ((RPV * j + rv) * (uint32_t)a.cache_row_stride + 8 * (cv ^ vswz(RPV * j + rv))));
  // A group that lies between the first and the last key that are seen needs no address of its own per row and tile: offsets made once
  // here, the page's address in scalars.  (With 64-bit products and clamps for each row of each tile, and the maxima exchanged through
  // LDS, 57.0 us where 55.0 now.  What is clamped, or rows of which 16 reach past 32 bits, in bytes, still goes that way.)
  const bool near_rows = a.cache_row_stride >= 0 && a.cache_row_stride < (1 << 26);
  auto bring = [&](int t, int img) __attribute__((always_inline)) {
    const int key0 = min(max(t * KT + 16 * wave, k_first & ~15), k_last), r_min = k_first - key0, r_max = k_last - key0;
    const int page = bshift >= 0 ? key0 >> bshift : key0 / bs;
    const int64_t off = (int64_t)table[page] * a.cache_block_stride + (int64_t)(key0 - page * bs) * a.cache_row_stride;
    const uint32_t kd = lds0 + (uint32_t)(img * IMG + 16 * wave * RSK), vd = lds0 + (uint32_t)(img * IMG + KTILE + 16 * wave * RSV);
    const u16 *kb = kc + off, *vb = vc + off;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    // (m0, the LDS address of the transfer, is a reserved register: nothing else in this kernel uses it)
    if (near_rows && r_min <= 0 && r_max >= 15) {      // nothing to clamp
#pragma unroll
      for (int j = 0; j < 16 / RPK; ++j)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(ko[j]), "s"(kb), "s"(__builtin_amdgcn_readfirstlane(kd + 1024u * j)) : "memory", "m0");
#pragma unroll
      for (int j = 0; j < 16 / RPV; ++j)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(vo[j]), "s"(vb), "s"(__builtin_amdgcn_readfirstlane(vd + 1024u * j)) : "memory", "m0");
      return;
    }
#pragma unroll
    for (int j = 0; j < 16 / RPK; ++j) {
      const int rr = RPK * j + rk;
      const u16* from = kb + (int64_t)max(min(rr, r_max), r_min) * a.cache_row_stride + 8 * (ck ^ kswz(rr));
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(__builtin_amdgcn_readfirstlane(kd + 1024u * j)) : "memory", "m0");
    }
#pragma unroll
    for (int j = 0; j < 16 / RPV; ++j) {
      const int rr = RPV * j + rv;
      const u16* from = vb + (int64_t)max(min(rr, r_max), r_min) * a.cache_row_stride + 8 * (cv ^ vswz(rr));
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(__builtin_amdgcn_readfirstlane(vd + 1024u * j)) : "memory", "m0");
    }
#pragma clang diagnostic pop
  };
  if (t_first + group <= t_last) bring(t_first + group, 0);
  // the queries (B operand): row c, columns 16 ks + 8 hi ..
  u16x8 qf[KS];
  {
    const u16* qg = (const u16*)a.q + ((int64_t)(q0 + tok) * a.n_heads + head) * D + 8 * hi;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const u16x8*>(qg + 16 * ks);
    // (they are there before the loop: a wait for them inside it would be one for the tile on its way)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[ks]));
  }
  // scores in units of log2: z = scale2 s - slope2 (pos - key), or under a cap cap2 tanh(s hsc / cap) in its place
  constexpr float kLog2e = 1.4426950408889634f;
  const float hsc = a.head_scale ? a.scale * a.head_scale[head] : a.scale;
  const float slope2 = MODS && a.slopes ? a.slopes[head] * kLog2e : 0.f;
  const bool cap = MODS && a.softcap > 0.f;
  const float cap2 = cap ? a.softcap * kLog2e : 0.f;
  float scale2 = cap ? hsc / a.softcap : hsc * kLog2e;
  if (!MODS) {             // (a maximum of scores is one of scaled scores where the scale is positive; -inf times it stays -inf)
    if (scale2 < 0.f) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[ks] ^= (u16)0x8000;
    }
    scale2 = fabsf(scale2) < 1e-30f ? 1e-30f : fabsf(scale2);      // (not fmaxf: what is not a number stays so)
  }

  f32x16 acc[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
  float m = HX_NEG_BIG, l = 0.f;
  // the transposing reads of V: lane 4 q + p of every 16 lanes brings row q, columns 16 half + 4 p ..
  const int tr_q = (lane & 15) >> 2, tr_x = vswz(tr_q) >> 2;
  const int tr_off = (4 * hi + tr_q) * RSV + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
  auto tile_step = [&](int t, int img) __attribute__((always_inline)) {
    const char* kt = smem_w + (2 * group + img) * IMG;
    const char* vt = kt + KTILE;
    f32x16 s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[u][e] = 0.f;
    {
      // the keys' fragments of the first half before its products, those of the second under them
      const char* krd = kt + c * RSK;
      const int kz = kswz(c);
      u16x8 ka[KS], kb[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) ka[ks] = *reinterpret_cast<const u16x8*>(krd + 16 * ((2 * ks + hi) ^ kz));
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        kb[ks] = *reinterpret_cast<const u16x8*>(krd + 32 * RSK + 16 * ((2 * ks + hi) ^ kz));
        s[0] = mma32(ka[ks], qf[ks], s[0]);
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s[1] = mma32(kb[ks], qf[ks], s[1]);
      __builtin_amdgcn_sched_group_barrier(0x100, KS, 0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, KS, 0);
    }
    // element e of half u: key t KT + 32 u + (e & 3) + 8 (e >> 2) + 4 hi
    const int key_l = t * KT + 4 * hi;
    float unit = scale2;                     // what a score still has to be multiplied by
    if (MODS) {
      unit = 1.f;
      if (cap) {
#pragma unroll
        for (int u = 0; u < 2; ++u) cap_scores<16>(s[u], scale2, cap2);
      } else {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int e = 0; e < 16; ++e) s[u][e] *= scale2;
      }
      if (a.slopes) {
        const float near = (float)(key_l - pos);             // (the distance itself is exact: a key at distance 0 loses nothing)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int e = 0; e < 16; ++e) s[u][e] = __builtin_fmaf(slope2, near + (float)(32 * u + (e & 3) + 8 * (e >> 2)), s[u][e]);
      }
    }
    if (!(t * KT + KT - 1 <= wpos0 && t * KT >= wlo1)) {      // (else every row of the wave sees the whole tile)
      const int last = pos - key_l, first = lo - key_l;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int k = 32 * u + (e & 3) + 8 * (e >> 2);
          if (k > last || k < first) s[u][e] = -INFINITY;
        }
    }
    // The weights refer to the largest score so far, half a tile at a time: its own is then 1, which no rounding to bfloat16 touches.  In
    // launches of few rows (FINE) they refer to the largest of these 32 keys, and what they add is scaled behind the products: the tile
    // form deals such a launch's keys to more waves, each with a largest score that weighs exactly 1.
    float m_ref[2] = {HX_NEG_BIG, HX_NEG_BIG}, m_new[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int e = 0; e < 16; ++e) m_ref[u] = fmaxf(m_ref[u], s[u][e]);
      m_ref[u] = halves_max(m_ref[u]) * unit;
      asm("" : "+v"(m_ref[u]));              // (rounded: left inside a difference below it would not be m_new's number)
      m_new[u] = fmaxf(u ? m_new[0] : m, m_ref[u]);
      if (!FINE) m_ref[u] = m_new[u];
    }
    u16x8 pf[2][2];
    float ps[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float pa = 0.f, pb = 0.f;
#pragma unroll
      for (int e = 0; e < 16; e += 2) {
        const float e0 = fast_exp2(__builtin_fmaf(s[u][e], unit, -m_ref[u])), e1 = fast_exp2(__builtin_fmaf(s[u][e + 1], unit, -m_ref[u]));
        pa += e0;
        pb += e1;
        pf[u][e >> 3][e & 7] = BF16::from_float(e0);
        pf[u][e >> 3][(e & 7) + 1] = BF16::from_float(e1);
      }
      ps[u] = pa + pb;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float alpha = fast_exp2(m - m_new[u]), beta = fast_exp2(m_ref[u] - m_new[u]);
      if (FINE || __builtin_amdgcn_ballot_w64(m_new[u] > m)) {
        l *= alpha;
        if constexpr (!FINE) {
#pragma unroll
          for (int i = 0; i < NDB; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][e] *= alpha;
        }
        m = m_new[u];
      }
      l = FINE ? __builtin_fmaf(ps[u], beta, l) : l + ps[u];
      auto product = [&](int db, int k2, f32x16 c) __attribute__((always_inline)) {
        const char* vrd = vt + (32 * u + 16 * k2) * RSV + tr_off;
        const u16x4 x0 = lds_tr_read(vrd + 64 * (db ^ tr_x)), x1 = lds_tr_read(vrd + 8 * RSV + 64 * (db ^ tr_x));
        return mma32(u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]}, pf[u][k2], c);
      };
      if constexpr (FINE) {
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
          f32x16 o;
#pragma unroll
          for (int e = 0; e < 16; ++e) o[e] = 0.f;
          o = product(db, 1, product(db, 0, o));
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[db][e] = __builtin_fmaf(o[e], beta, acc[db][e] * alpha);
        }
      } else {
#pragma unroll
        for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
          for (int db = 0; db < NDB; ++db) acc[db] = product(db, k2, acc[db]);
      }
    }
  };
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int t0 = t_first; t0 <= t_last; t0 += KG) {
    const int t = t0 + group, img = (t0 - t_first) / KG & 1;
    if (t + KG <= t_last) bring(t + KG, img ^ 1);
    if (live && t <= t_last && t * KT <= wpos1 && t * KT + KT - 1 >= wlo0) tile_step(t, img);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this wave's part of the next tile is there
    __syncthreads();                                       // everybody's is, and this one has been read
  }
  // Two groups: each hands the other half of its columns and finishes the rest.  (One tile: the first group has it all.)
  const bool two = KG > 1 && t_last > t_first;
  if constexpr (KG > 1) {
    if (two) {
      f32x4* part = reinterpret_cast<f32x4*>(smem_w + 2 * IMG) + wave * (4 * NDB + 1) * 64 + lane;
      auto hand = [&](auto first) __attribute__((always_inline)) {      // (first: the first column block that the other group finishes)
#pragma unroll
        for (int i = 0; i < NDB / 2; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const f32x16& x = acc[first + i];
            part[(4 * (first + i) + e) * 64] = f32x4{x[4 * e], x[4 * e + 1], x[4 * e + 2], x[4 * e + 3]};
          }
      };
      float2* ml = reinterpret_cast<float2*>(part - lane + 4 * NDB * 64) + lane;
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
        for (int i = 0; i < NDB / 2; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            f32x16& x = acc[first + i];
            const f32x4 y = part[(4 * (first + i) + e) * 64];
#pragma unroll
            for (int k = 0; k < 4; ++k) x[4 * e + k] = __builtin_fmaf(x[4 * e + k], mine, y[k] * theirs);
          }
      };
      if (group) take(std::integral_constant<int, NDB / 2>());
      else take(std::integral_constant<int, 0>());
    } else if (group) {
      return;
    }
  }
  if (!live && !two) return;
  // out, through LDS (the images are free): whole rows a store.  O[row c][column 32 db + 8 (e >> 2) + 4 hi + (e & 3)]
  float total = l + __shfl_xor(l, 32, 64);
  if (a.sinks) total += fast_exp2(a.sinks[head] * kLog2e - m);      // the sink: one more term, without a value
  const float inv = 1.0f / total;
  char* ob = smem_w + wave * 32 * RSV;
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
    if (two && (db < NDB / 2) == (group != 0)) continue;
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4) {
      u16x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = BF16::from_float(acc[db][4 * e4 + i] * inv);
      *reinterpret_cast<u16x4*>(ob + c * RSV + (((8 * db + 2 * e4 + hi) ^ (c & (LV - 1))) << 3)) = o;
    }
  }
  if (two) __syncthreads();
  else wave_lds_sync();
#pragma unroll
  for (int j = 0; j < 32 / RPV; ++j) {
    if (two && (j & 1) != group) continue;
    const int rl = RPV * j + rv, ro = row0 + rl;
    // 8-byte slots 2 ch, 2 ch + 1 of row rl sit in chunk ch ^ (rl' >> 1), in turned order when rl' is odd (rl' = rl mod V / 8)
    u16x8 v = *reinterpret_cast<const u16x8*>(ob + rl * RSV + 16 * (cv ^ ((rl & (LV - 1)) >> 1)));
    if (rl & 1) v = u16x8{v[4], v[5], v[6], v[7], v[0], v[1], v[2], v[3]};
    if (ro >= 0) *reinterpret_cast<u16x8*>((u16*)a.out + ((int64_t)(q0 + ro / R) * a.n_heads + kvh * R + ro % R) * V + 8 * cv) = v;
  }
}

template <int D, int V>
int launch_wide(const hxm_biased_attn_args& a, hipStream_t s) {
  // row tiles of all sequences, at most
  const int R = a.n_heads / a.kv_heads;
  const int64_t slots = ((int64_t)a.n_tokens * R + 127) / 128 + a.n_seq, grid = (slots * a.kv_heads + 7) / 8 * 8;
  if (grid > 0x7fffffff) return HX_ERR_SHAPE;
  const bool mods = a.slopes || a.softcap > 0.f;
  // few rows: fewer tiles of 16 than the waves that the tile form's keys are dealt to (see its callers)
  const bool fine = (int64_t)a.n_seq * a.kv_heads * (((int64_t)a.max_q_len * R + 15) / 16) < 2048;
  // A workgroup a compute unit: two groups of waves share its keys, so that a SIMD has two waves.  Portions of up to a tile's keys have nothing to
  // share (us, one group and two: 4 of 20 - 52 tokens, cap and slopes 10.6 11.6; one of 128 - 152, 10.4 10.6; 2 of 81 - 217 18.1 16.2, 1082 behind 463 41.8
  // 33.4, 110 behind 495 25.5 19.7; by the number of workgroups 140 - 256 3 - 25 % faster, 272 20.5 28.4 under a short window, 280 37.1 28.9, 288, of 24 portions
  // of 78, 16.6 22.5, 320 18.8 28.1 and 28.4 28.6, 600 - 1000 12 - 25 % slower).  The portions' last row tiles are half full in the mean; equal portions are
  // counted as they are (12 of 67 tokens in 288 workgroups 10.3 12.9).
  int64_t workgroups = ((int64_t)a.n_tokens * R / 64 + a.n_seq) * a.kv_heads / 2;
  if (a.n_tokens == (int64_t)a.n_seq * a.max_q_len) workgroups = std::max(workgroups, a.n_seq * (((int64_t)a.max_q_len * R + 127) / 128) * a.kv_heads);
  const bool two = a.max_q_len > 64 && workgroups <= 256;
  auto kernel = two ? (fine ? (mods ? biased_attn_wide_kernel<D, V, true, true, 2> : biased_attn_wide_kernel<D, V, false, true, 2>)
                            : (mods ? biased_attn_wide_kernel<D, V, true, false, 2> : biased_attn_wide_kernel<D, V, false, false, 2>))
                    : (fine ? (mods ? biased_attn_wide_kernel<D, V, true, true, 1> : biased_attn_wide_kernel<D, V, false, true, 1>)
                            : (mods ? biased_attn_wide_kernel<D, V, true, false, 1> : biased_attn_wide_kernel<D, V, false, false, 1>));
  constexpr size_t images = 2 * 64 * (2 * D + 2 * V), part = 4 * (V / 2 + 4) * 256;      // (of a group of waves; what the groups hand over, in the place of the second one's images)
  const size_t lds = two ? images + std::max(images, part) : images;
  if (lds > 48 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
      hxm::last_hip_error() = (int)e;
      return HX_ERR_HIP;
    }
  }
  kernel<<<dim3((unsigned)grid), dim3(two ? 512 : 256), lds, s>>>(a, (int)slots);
  return hxm::check_launch();
}

// ---------------------------------------------------------------------------------------------------------------
// Step form (bfloat16, fewer than 64 rows of a key head or few row tiles behind many keys, key and value heads of 64 or 128,
// pages of whole 16-row groups): a wave takes 16 rows of ONE (sequence, key head) and one run of its keys, in tiles of 32.  Bound by memory: the
// tile form asks for a key's row in 64-byte pieces, sixteen rows an instruction, and has one chunk in flight; here rows go whole
// from the paged cache to LDS, the next tile's while this one's are awaited — no register holds them and no barrier is needed.
// A wave's two images are 32 KB of LDS at heads of 128 (64: 16): five waves a compute unit by themselves, one workgroup of four.  Products are 16 x 16 x 32 and swapped, S^T = K Q^T,
// O^T += V^T P^T: a row of the softmax is one lane, its weights stay in their registers.  16-byte chunk x of row r sits at
// x ^ swz(r): rows r and 15 - r share a 32-byte place (their chunks turned), so that a pass of a 16-byte read and a transposing
// read (eight rows, 32 bytes each) both reach every bank once.
// Two or four runs of a row tile's keys are a workgroup's, a wave each, merged through LDS where the images were; only more of them, and three or seven, go
// through memory and a second launch.  32 tokens of 1025 - 2047 keys 46.7 us with that launch, 43 in workgroups of four, 20 of 55 - 253 9.6 and 6.7, 224 row tiles of
// 1500 45.9 (five splits) and 35.3; 15 % in the mean of 50 batches.
// Measured, 32 heads of 128 on 8 key heads: 32 tokens of 1025 - 2047 keys 56 us in the tile form and its merge, 43 here (4.7 TB/s, with the way to the first
// keys); by single waves and the launch that merges: 128 tokens of 500 - 1500 keys 163 us and 109; 32 tokens, 2 key heads 57 us and 24; 16 tokens behind 4000 keys
// 93 us (tile), 79 (wide) and 29.
// ---------------------------------------------------------------------------------------------------------------
template <int D, int V, bool MODS, int W>      // MODS: slopes or a soft cap; W: waves, a split each
__global__ __launch_bounds__(64 * W) void biased_attn_step_kernel(hxm_biased_attn_args a, int tiles_per_seq) {
  constexpr int KT = 32, KS = D / 32, NDB = V / 16, RSK = 2 * D, RSV = 2 * V, LK = D / 8, LV = V / 8;
  constexpr int KTILE = KT * RSK, IMG = KTILE + KT * RSV, NLK = 16 * LK / 64, NLV = 16 * LV / 64;      // transfers of 16 rows
  extern __shared__ __attribute__((aligned(256))) char smem_s[];       // [W][2][K rows | V rows]
  auto swz = [](int row, bool full) {        // full: rows of whole bank rows, 16 places of a chunk, else 8 for each parity of the row
    if (full) return (row & 15) < 8 ? 2 * (row & 7) : 31 - 2 * (row & 15);
    const int h = (row & 15) >> 1;
    return h < 4 ? 2 * h : 15 - 2 * h;
  };
  typedef __attribute__((address_space(4))) const int32_t c_i32;       // (uniform indices: through the scalar cache)
  const int G = a.kv_heads, R = a.n_heads / a.kv_heads, n_splits = a.n_splits > 1 ? a.n_splits : 1;
  // workgroup -> (sequence, row tile, split, key head), key heads fastest: the rows of a page are asked for at about one time
  int at = blockIdx.x;
  const int kvh = at % G;
  at /= G;
  const int wave = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0, n_groups = n_splits / W, group = at % n_groups;
  const int split = group * W + wave;
  at /= n_groups;
  const int tile = at % tiles_per_seq, b = at / tiles_per_seq;
  const int q0 = ((c_i32*)a.q_cu)[b], n_rows = (((c_i32*)a.q_cu)[b + 1] - q0) * R, n_tiles = (n_rows + 15) / 16;
  if (tile >= n_tiles) return;
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int row0 = n_rows - (n_tiles - tile) * 16;      // (row tiles end with the portion; rows below 0 do not exist)
  const int r = max(row0 + c, 0), tok = r / R, head = kvh * R + r % R;
  const int pos = a.positions[q0 + tok], lo = first_visible(pos, a.mask_kind, a.mask_size);
  const int pos_min = wave_min_int(pos), k_last = wave_max_int(pos), k_first = wave_min_int(lo), lo_max = wave_max_int(lo);
  int t_first = k_first / KT, t_last = k_last < 0 ? t_first - 1 : k_last / KT;      // (positions below 0 see nothing)
  if (n_splits > 1) {                        // this split's run of tiles (the last splits may get none)
    const int per = (t_last - t_first + n_splits) / n_splits;
    t_first += split * per;
    t_last = min(t_last, t_first + per - 1);
  }
  u16x8 qf[KS];                              // the queries (B operand): row c, columns 32 ks + 8 g ..
  {
    const u16* qg = (const u16*)a.q + ((int64_t)(q0 + tok) * a.n_heads + head) * D + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const u16x8*>(qg + 32 * ks);
  }
  constexpr float kLog2e = 1.4426950408889634f;
  float hsc = a.head_scale ? a.scale * a.head_scale[head] : a.scale;
  float slope2 = MODS && a.slopes ? a.slopes[head] * kLog2e : 0.f;
  float sink2 = a.sinks ? a.sinks[head] * kLog2e : -INFINITY;
  const int32_t* table = a.block_table + ((c_i32*)a.cu_block_lens)[b];
  const int bs = a.block_size, bshift = (bs & (bs - 1)) == 0 ? __ffs(bs) - 1 : -1;
  auto page_of = [&](int key) { return bshift >= 0 ? key >> bshift : key / bs; };
  // The key that a group of 16 is brought from on.  What lies in front of the first key that some row sees, or behind the last, is not
  // touched (its page may be gone): rows there repeat that key, masked.
  const int k_from = k_first & ~15;
  auto group_key = [&](int group) { return min(max(16 * group, k_from), k_last); };
  // lane i: the page of the i-th group of 16 keys from group pages0 on
  int pages0 = 2 * t_first, pages = k_last < 0 ? 0 : table[page_of(group_key(pages0 + lane))];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[ks]));
  asm volatile("" : "+v"(pages), "+v"(hsc), "+v"(slope2), "+v"(sink2));      // (all there before the transfers start: a wait for them would be one for those)
  const u16* kc = (const u16*)a.key_cache + (int64_t)kvh * a.head_stride;
  const u16* vc = (const u16*)a.value_cache + (int64_t)kvh * a.head_stride;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem_s + (uint32_t)(wave * 2 * IMG);
  const uint32_t row_bytes = (uint32_t)(2 * a.cache_row_stride);
  auto bring = [&](int t, int img) __attribute__((always_inline)) {
    if (2 * t + 1 - pages0 > 63) {
      pages0 = 2 * t;
      pages = table[page_of(group_key(pages0 + lane))];
      asm volatile("" : "+v"(pages));        // (waited for here: after the branch it would be a wait in every tile)
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (the reads of the image that this replaces are done)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    // (m0, the LDS address of the transfer, is a reserved register: nothing else in this kernel uses it)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int key0 = group_key(2 * t + u), r_min = k_first - key0, r_max = k_last - key0;
      const int64_t off = (int64_t)__builtin_amdgcn_readlane(pages, 2 * t + u - pages0) * a.cache_block_stride +
                          (int64_t)(key0 - page_of(key0) * bs) * a.cache_row_stride;
      const uint32_t kd = lds0 + (uint32_t)(img * IMG + 16 * u * RSK), vd = lds0 + (uint32_t)(img * IMG + KTILE + 16 * u * RSV);
#pragma unroll
      for (int j = 0; j < NLK; ++j) {
        const int rr = (64 * j + lane) / LK, ch = (64 * j + lane) % LK;
        const uint32_t from = (uint32_t)max(min(rr, r_max), r_min) * row_bytes + 16u * (uint32_t)(ch ^ swz(rr, D == 128));
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(from), "s"(kc + off), "s"(__builtin_amdgcn_readfirstlane(kd + 1024u * j)) : "memory", "m0");
      }
#pragma unroll
      for (int j = 0; j < NLV; ++j) {
        const int rr = (64 * j + lane) / LV, ch = (64 * j + lane) % LV;
        const uint32_t from = (uint32_t)max(min(rr, r_max), r_min) * row_bytes + 16u * (uint32_t)(ch ^ swz(rr, V == 128));
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(from), "s"(vc + off), "s"(__builtin_amdgcn_readfirstlane(vd + 1024u * j)) : "memory", "m0");
      }
    }
#pragma clang diagnostic pop
  };
  if (t_first <= t_last) bring(t_first, 0);
  // scores in units of log2: z = scale2 s - slope2 (pos - key), or under a cap cap2 tanh(s hsc / cap) in its place
  const bool cap = MODS && a.softcap > 0.f;
  const float cap2 = cap ? a.softcap * kLog2e : 0.f;
  float scale2 = cap ? hsc / a.softcap : hsc * kLog2e;
  if (!MODS) {             // (a maximum of scores is one of scaled scores where the scale is positive; -inf times it stays -inf)
    if (scale2 < 0.f) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[ks] ^= (u16)0x8000;
    }
    scale2 = fabsf(scale2) < 1e-30f ? 1e-30f : fabsf(scale2);      // (not fmaxf: what is not a number stays so)
  }
  f32x4 acc[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = HX_NEG_BIG, l = 0.f;
  // Reads of rows: chunk 4 ks + g of row c.  Transposing reads: lane 4 q + p of a group of 16 brings row 4 g + q (and the row 16
  // below it: the same place), columns 16 db + 4 p ..: chunk 2 db + p / 2.
  const uint32_t kp0 = lds0 + (uint32_t)(c * RSK + 16 * (g ^ swz(c, D == 128)));
  const uint32_t vp0 = lds0 + (uint32_t)(KTILE + (4 * g + (c >> 2)) * RSV + 16 * (((c & 3) >> 1) ^ swz(4 * g + (c >> 2), V == 128)) + 8 * (c & 1));
  auto row_read = [](uint32_t from) __attribute__((always_inline)) {
    return *reinterpret_cast<__attribute__((address_space(3))) const u16x8*>((uintptr_t)from);
  };
  auto tr_read = [](uint32_t from) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) hx_s16x4_t lds_s4;
    return __builtin_bit_cast(u16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(uintptr_t)from));
  };
  for (int t = t_first; t <= t_last; ++t) {
    const int img = (t - t_first) & 1, key0 = t * KT;
    if (t < t_last) {
      bring(t + 1, img ^ 1);
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (NLK + NLV)) : "memory");      // this tile is there, the next on its way
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    const uint32_t kp = kp0 + (uint32_t)(img * IMG), va = vp0 + (uint32_t)(img * IMG);
    f32x4 s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) s[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int u = 0; u < 2; ++u) s[u] = Mfma<BF16>::mma(row_read((kp ^ (64u * ks)) + 16u * u * RSK), qf[ks], s[u]);
    const int key_l = key0 + 4 * g;          // element e of half u: key key_l + 16 u + e
    float unit = scale2;                     // what a score still has to be multiplied by
    if (MODS) {
      unit = 1.f;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (cap) cap_scores<4>(s[u], scale2, cap2);
        else s[u] *= scale2;
      }
      if (a.slopes) {
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e >> 2][e & 3] += slope2 * (float)(key_l + 16 * (e >> 2) + (e & 3) - pos);
      }
    }
    float mx = HX_NEG_BIG;
    if (key0 + KT - 1 <= pos_min && key0 >= lo_max) {      // every row of the wave sees all of them
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
    // A tile's weights refer to the tile's own largest score, which is then 1 and which no rounding to bfloat16 touches; what the tile
    // adds is scaled behind its products.  (Bound by memory, this costs nothing; with weights that refer to the largest score so far and
    // half as many splits as the tile form took, 32 tokens of 1025 - 2047 keys were off by 2.17e-3 of the result, 2.13 in the tile form.)
    float m_tile = groups_max(mx) * unit;
    asm("" : "+v"(m_tile));                  // (rounded: left inside the difference below it would not be m_new's number)
    const float m_new = fmaxf(m, m_tile);
    const float alpha = fast_exp2(m - m_new), beta = fast_exp2(m_tile - m_new);
    m = m_new;
    u16x8 pf;
    float l_tile = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float p = fast_exp2(__builtin_fmaf(s[e >> 2][e & 3], unit, -m_tile));
      l_tile += p;
      pf[e] = BF16::from_float(p);
    }
    l = __builtin_fmaf(l, alpha, l_tile * beta);
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      const u16x4 x0 = tr_read(va ^ (32u * db)), x1 = tr_read((va ^ (32u * db)) + 16u * RSV);
      const f32x4 o = Mfma<BF16>::mma(u16x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]}, pf, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[db][e] = __builtin_fmaf(o[e], beta, acc[db][e] * alpha);
    }
    // (reads stay a few products ahead)
    constexpr int kAhead = NDB < 6 ? NDB : 6;
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kAhead, 0);
#pragma unroll
    for (int i = 0; i < NDB - kAhead; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kAhead, 0);
  }
  float total = l + __shfl_xor(l, 16, 64);
  total += __shfl_xor(total, 32, 64);
  constexpr int NW = NDB / W;                // column blocks that a wave finishes
  if constexpr (W > 1) {                     // the waves' splits merged, each wave's part where its images were
    f32x4* part = reinterpret_cast<f32x4*>(smem_s);
    auto part_of = [&](int w) { return part + w * (2 * IMG / 16); };
#pragma unroll
    for (int db = 0; db < NDB; ++db) part_of(wave)[64 * db + lane] = acc[db];
    reinterpret_cast<float2*>(part_of(wave) + 64 * NDB)[lane] = float2{m, total};
    __syncthreads();
    float2 ml[W];
    f32x4 v[W][NW];
#pragma unroll
    for (int w = 0; w < W; ++w) {
      ml[w] = reinterpret_cast<const float2*>(part_of(w) + 64 * NDB)[lane];
#pragma unroll
      for (int i = 0; i < NW; ++i) v[w][i] = part_of(w)[64 * (NW * wave + i) + lane];
    }
    m = ml[0].x;
#pragma unroll
    for (int w = 1; w < W; ++w) m = fmaxf(m, ml[w].x);
    total = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float weight = fast_exp2(ml[w].x - m);
      total += weight * ml[w].y;
#pragma unroll
      for (int i = 0; i < NW; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][e] += weight * v[w][i][e];
    }
  }
  if (row0 + c < 0) return;                  // (rows below 0 are whole columns of lanes)
  const int col0 = 16 * NW * wave;
  if (n_groups > 1) {
    // what this split adds to a row, not normalised: ws_o [sequence, key head, tile][row][split][V], ws_ml [..][split][maximum (log2), sum]
    const size_t slot = ((((size_t)b * G + kvh) * tiles_per_seq + tile) * 16 + c) * n_groups + group;
    float* wo = a.ws_o + slot * V + col0 + 4 * g;
#pragma unroll
    for (int db = 0; db < NW; ++db) *reinterpret_cast<f32x4*>(wo + 16 * db) = acc[db];
    if (g == 0 && wave == 0) {
      a.ws_ml[2 * slot] = m;
      a.ws_ml[2 * slot + 1] = total;
    }
    return;
  }
  const float inv = 1.0f / (total + fast_exp2(sink2 - m));      // the sink: one more term, without a value
  u16* og = (u16*)a.out + ((int64_t)(q0 + tok) * a.n_heads + head) * V + col0 + 4 * g;
#pragma unroll
  for (int db = 0; db < NW; ++db)
    *reinterpret_cast<u16x4*>(og + 16 * db) = u16x4{BF16::from_float(acc[db][0] * inv), BF16::from_float(acc[db][1] * inv), BF16::from_float(acc[db][2] * inv), BF16::from_float(acc[db][3] * inv)};
}

// The splits of a row merged: out = sum_s O_s 2^(m_s - M) / sum_s l_s 2^(m_s - M).  A row to V / 4 lanes; one pass over the splits,
// four at a time, their loads all in flight together.
template <int V>
__global__ __launch_bounds__(256) void biased_attn_merge_kernel(hxm_biased_attn_args a, int n_parts, int tiles_per_seq) {
  const int64_t at = (int64_t)blockIdx.x * 256 + threadIdx.x, slot = at / (V / 4);      // slot: row c of (sequence, key head, tile)
  const int G = a.kv_heads, R = a.n_heads / a.kv_heads, NS = n_parts, col = 4 * (int)(at % (V / 4));
  const int64_t item = slot / 16;
  const int tile = (int)(item % tiles_per_seq), kvh = (int)(item / tiles_per_seq % G), b = (int)(item / tiles_per_seq / G);
  if (b >= a.n_seq) return;
  const int q0 = a.q_cu[b], n_rows = (a.q_cu[b + 1] - q0) * R, n_tiles = (n_rows + 15) / 16;
  const int r = n_rows - (n_tiles - tile) * 16 + (int)(slot % 16);
  if (tile >= n_tiles || r < 0) return;
  const int head = kvh * R + r % R;
  const float* ml = a.ws_ml + 2 * slot * NS;
  const float* wo = a.ws_o + slot * NS * V + col;
  const float sink2 = a.sinks ? a.sinks[head] * 1.4426950408889634f : -INFINITY;
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
      v[i] = *reinterpret_cast<const f32x4*>(wo + (size_t)s * V);
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
  const float inv = 1.0f / (total + fast_exp2(sink2 - M));      // the sink counts once, here
  u16* og = (u16*)a.out + ((int64_t)(q0 + r / R) * a.n_heads + head) * V + col;
  *reinterpret_cast<u16x4*>(og) = u16x4{BF16::from_float(o[0] * inv), BF16::from_float(o[1] * inv), BF16::from_float(o[2] * inv), BF16::from_float(o[3] * inv)};
}

template <int D, int V, int W>
int launch_step_waves(const hxm_biased_attn_args& a, hipStream_t s) {
  const int R = a.n_heads / a.kv_heads, tiles_per_seq = (int)(((int64_t)a.max_q_len * R + 15) / 16), n_groups = (a.n_splits > 1 ? a.n_splits : 1) / W;
  const int64_t items = (int64_t)a.n_seq * a.kv_heads * tiles_per_seq;
  if (items * n_groups > 0x7fffffff) return HX_ERR_SHAPE;
  const bool mods = a.slopes || a.softcap > 0.f;
  auto kernel = mods ? biased_attn_step_kernel<D, V, true, W> : biased_attn_step_kernel<D, V, false, W>;
  constexpr size_t lds = (size_t)W * 2 * 32 * (2 * D + 2 * V);
  if (lds > 48 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
      hxm::last_hip_error() = (int)e;
      return HX_ERR_HIP;
    }
  }
  kernel<<<dim3((unsigned)(items * n_groups)), dim3(64 * W), lds, s>>>(a, tiles_per_seq);
  if (n_groups > 1) biased_attn_merge_kernel<V><<<dim3((unsigned)((items * 16 * (V / 4) + 255) / 256)), dim3(256), 0, s>>>(a, n_groups, tiles_per_seq);
  return hxm::check_launch();
}
// A few workgroups of four waves more than compute units take as long as twice as many: waves by themselves then (288 row tiles of 700 - 2100 keys 52.6 us,
// by fours 55.8)
bool between_rounds(int64_t tiles) { return tiles > 256 && tiles < 384; }
template <int D, int V>
int launch_step(const hxm_biased_attn_args& a, hipStream_t s) {
  const int64_t tiles = (int64_t)a.n_seq * a.kv_heads * (((int64_t)a.max_q_len * (a.n_heads / a.kv_heads) + 15) / 16);
  if (a.n_splits == 4 && between_rounds(tiles)) return launch_step_waves<D, V, 1>(a, s);
  if (a.n_splits > 1 && a.n_splits % 4 == 0) return launch_step_waves<D, V, 4>(a, s);
  if (a.n_splits > 1 && a.n_splits % 2 == 0) return launch_step_waves<D, V, 2>(a, s);
  return launch_step_waves<D, V, 1>(a, s);
}

// the splits of a (sequence, kv head, row tile) merged: out = sum_s O_s e^(m_s - M) / sum_s l_s e^(m_s - M)
__global__ __launch_bounds__(256) void biased_attn_combine_kernel(hxm_biased_attn_args a, int tiles_per_seq) {
  const int64_t item = blockIdx.x;
  const int G = a.kv_heads, R = a.n_heads / a.kv_heads, V = a.vdim, V16 = (V + 15) / 16 * 16, NS = a.n_splits;
  const int tile = (int)(item % tiles_per_seq);
  const int kvh = (int)((item / tiles_per_seq) % G);
  const int b = (int)(item / ((int64_t)tiles_per_seq * G));
  const int q0 = a.q_cu[b];
  const int n_rows = (a.q_cu[b + 1] - q0) * R;
  if (tile * 16 >= n_rows) return;
  __shared__ float wgt[16][65];      // [row][split] weight e^(m_s - M) / L (NS <= 64)
  if (threadIdx.x < 16) {
    const int row = threadIdx.x;
    const float* wml = a.ws_ml + (size_t)item * NS * 32;
    float M = -1.0e30f;
    for (int s = 0; s < NS; ++s) M = fmaxf(M, wml[s * 32 + 2 * row]);
    float L = 0.f;
    for (int s = 0; s < NS; ++s) L += wml[s * 32 + 2 * row + 1] * __expf(wml[s * 32 + 2 * row] - M);
    if (a.sinks) L += expf(a.sinks[kvh * R + (tile * 16 + row) % R] - M);      // the sink counts once, here
    const float inv = L > 0.f ? 1.0f / L : 0.f;
    for (int s = 0; s < NS; ++s) wgt[row][s] = __expf(wml[s * 32 + 2 * row] - M) * inv;
  }
  __syncthreads();
  const float* wo = a.ws_o + (size_t)item * NS * 16 * V16;
  for (int e = threadIdx.x; e < 16 * V; e += 256) {
    const int row = e / V, col = e % V;
    const int r = tile * 16 + row;
    if (r >= n_rows) continue;
    float v = 0.f;
    for (int s = 0; s < NS; ++s) v += wo[((size_t)s * 16 + row) * V16 + col] * wgt[row][s];
    ((u16*)a.out)[((int64_t)(q0 + r / R) * a.n_heads + kvh * R + r % R) * V + col] = BF16::from_float(v);
  }
}

template <int KK>
int launch_tile(const hxm_biased_attn_args& a, hipStream_t s) {
  const size_t per_wave = (size_t)32 * (2 * (KK * 32) + 32) + 16 * kPStride * 2;
  int waves = 4;
  while (waves > 1 && per_wave * waves > 64 * 1024) waves >>= 1;
  const int R = a.n_heads / a.kv_heads;
  const int tiles_per_seq = (int)(((int64_t)a.max_q_len * R + 15) / 16);
  const int n_splits = a.n_splits > 1 ? a.n_splits : 1;
  if constexpr (KK <= 4) {
    if (n_splits == 1 && tiles_per_seq >= 4 && a.form != 2) {      // portions of prompts: four row tiles share every chunk
      const int groups_per_seq = (tiles_per_seq + 3) / 4;
      const size_t lds_g = (size_t)128 * (2 * (KK * 32) + 32) + 4 * 16 * kPStride * 2;
      biased_attn_group_kernel<KK><<<dim3((unsigned)((int64_t)a.n_seq * a.kv_heads * groups_per_seq)), dim3(256), lds_g, s>>>(a, groups_per_seq);
      return hxm::check_launch();
    }
  }
  const int64_t items = (int64_t)a.n_seq * a.kv_heads * tiles_per_seq;
  const dim3 grid((unsigned)((items * n_splits + waves - 1) / waves));
  biased_attn_tile_kernel<KK><<<grid, dim3(64 * waves), per_wave * waves, s>>>(a, tiles_per_seq, waves);
  if (n_splits > 1) biased_attn_combine_kernel<<<dim3((unsigned)items), dim3(256), 0, s>>>(a, tiles_per_seq);
  return hxm::check_launch();
}

bool tile_form_serves(const hxm_biased_attn_args& a) {
  const bool aligned = a.dim % 8 == 0 && a.vdim % 8 == 0 && a.head_stride % 8 == 0 && a.cache_row_stride % 8 == 0 &&
                       a.cache_block_stride % 8 == 0 && aligned16(a.key_cache) && aligned16(a.value_cache) && aligned16(a.q);
  return a.dtype == HX_BF16 && aligned && a.dim <= 256 && a.vdim <= 256 && a.q_cu && a.n_seq > 0 && a.max_q_len > 0 && a.form != 1;
}

}  // namespace

extern "C" int hxm_qk_norm_cache(const void* proj, int64_t proj_stride, int64_t q_off, int64_t q_size, int64_t k_off,
                                 int64_t k_size, int64_t v_off, int64_t v_size, const float* q_w, const float* k_w, float eps,
                                 void* q_out, const int32_t* slot_ids, void* key_cache, void* value_cache,
                                 int64_t cache_row_stride, int64_t head_stride, int32_t kv_heads, int64_t n_tokens, int dtype,
                                 void* stream) {
  if (n_tokens < 0 || q_size < 1 || k_size < 0 || v_size < 0 || kv_heads < 1) return HX_ERR_SHAPE;
  if (n_tokens == 0) return HX_OK;
  if (!proj || !q_out) return HX_ERR_NULL;
  if (k_size > 0) {
    if (!slot_ids || !key_cache || !value_cache) return HX_ERR_NULL;
    if (k_size % kv_heads || v_size % kv_heads || v_size < 1) return HX_ERR_SHAPE;
    if (k_size / kv_heads > head_stride || v_size / kv_heads > head_stride || cache_row_stride < head_stride * kv_heads) return HX_ERR_STRIDE;
  }
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)n_tokens), block(256);
  const uintptr_t es = dtype == HX_F32 ? 4 : 2;
  auto by4 = [&](const void* p) { return ((uintptr_t)p % (4 * es)) == 0; };
  int vec = q_off % 4 == 0 && q_size % 4 == 0 && proj_stride % 4 == 0 && by4(proj) && by4(q_out) &&
            (!q_w || (uintptr_t)q_w % 16 == 0);
  if (k_size > 0)
    vec = vec && k_off % 4 == 0 && v_off % 4 == 0 && (k_size / kv_heads) % 4 == 0 && (v_size / kv_heads) % 4 == 0 &&
          cache_row_stride % 4 == 0 && head_stride % 4 == 0 && by4(key_cache) && by4(value_cache) && (!k_w || (uintptr_t)k_w % 16 == 0);
  switch (dtype) {
    case HX_F32:
      qk_norm_cache_kernel<F32><<<grid, block, 0, s>>>((const float*)proj, proj_stride, q_off, q_size, k_off, k_size, v_off, v_size,
                                                       q_w, k_w, eps, (float*)q_out, slot_ids, (float*)key_cache, (float*)value_cache,
                                                       cache_row_stride, head_stride, kv_heads, vec);
      break;
    case HX_BF16:
      qk_norm_cache_kernel<BF16><<<grid, block, 0, s>>>((const u16*)proj, proj_stride, q_off, q_size, k_off, k_size, v_off, v_size,
                                                        q_w, k_w, eps, (u16*)q_out, slot_ids, (u16*)key_cache, (u16*)value_cache,
                                                        cache_row_stride, head_stride, kv_heads, vec);
      break;
    default: return HX_ERR_DTYPE;
  }
  return hxm::check_launch();
}

extern "C" int hxm_biased_attention(const hxm_biased_attn_args* args, void* stream) {
  if (!args) return HX_ERR_NULL;
  const hxm_biased_attn_args& a = *args;
  if (a.n_tokens < 0 || a.n_heads < 1 || a.kv_heads < 1 || a.n_heads % a.kv_heads || a.dim < 1 || a.vdim < 1 ||
      a.vdim > 64 * kMaxVCols || a.block_size < 1)
    return HX_ERR_SHAPE;
  if (a.mask_kind < HXM_MASK_CAUSAL || a.mask_kind > HXM_MASK_CHUNK || (a.mask_kind != HXM_MASK_CAUSAL && a.mask_size < 1)) return HX_ERR_SHAPE;
  if (a.n_tokens == 0) return HX_OK;
  if (!a.out || !a.q || !a.key_cache || !a.value_cache || !a.tok_seq || !a.positions || !a.block_table || !a.cu_block_lens) return HX_ERR_NULL;
  if (a.dim > a.head_stride || a.vdim > a.head_stride) return HX_ERR_STRIDE;
  hipStream_t s = (hipStream_t)stream;
  if (a.n_splits > 1 && (a.n_splits > 64 || !a.ws_o || !a.ws_ml || !tile_form_serves(a))) return HX_ERR_WORKSPACE;
  if (tile_form_serves(a)) {
    // heads of 64 or 128 over pages of whole 16-row groups: the wide form from half a row tile of 128 on, the step form below and
    // where the caller has the keys of a row tile dealt out (the tile form: other head and page sizes)
    const bool whole = (a.dim == 64 || a.dim == 128) && (a.vdim == 64 || a.vdim == 128) && a.form != 2 && a.block_size % 16 == 0 && aligned16(a.out);
    if (whole && a.n_splits <= 1 && (int64_t)a.max_q_len * (a.n_heads / a.kv_heads) >= 64) {
      if (a.dim == 64) return a.vdim == 64 ? launch_wide<64, 64>(a, s) : launch_wide<64, 128>(a, s);
      return a.vdim == 64 ? launch_wide<128, 64>(a, s) : launch_wide<128, 128>(a, s);
    }
    if (whole && a.cache_row_stride < (1 << 26) && aligned16(a.ws_o)) {
      if (a.dim == 64) return a.vdim == 64 ? launch_step<64, 64>(a, s) : launch_step<64, 128>(a, s);
      return a.vdim == 64 ? launch_step<128, 64>(a, s) : launch_step<128, 128>(a, s);
    }
    const int kk = ((a.dim > a.vdim ? a.dim : a.vdim) + 31) / 32;
    if (kk <= 1) return launch_tile<1>(a, s);
    if (kk <= 2) return launch_tile<2>(a, s);
    if (kk <= 4) return launch_tile<4>(a, s);
    return launch_tile<8>(a, s);
  }
  const int64_t items = (int64_t)a.n_tokens * a.n_heads;
  const size_t lds = 4 * ((size_t)a.dim + 64) * sizeof(float);
  if (lds > 64 * 1024) return HX_ERR_SHAPE;
  const dim3 grid((unsigned)((items + 3) / 4)), block(256);
  switch (a.dtype) {
    case HX_F32: biased_attn_rows_kernel<F32><<<grid, block, lds, s>>>(a); break;
    case HX_BF16: biased_attn_rows_kernel<BF16><<<grid, block, lds, s>>>(a); break;
    default: return HX_ERR_DTYPE;
  }
  return hxm::check_launch();
}

// Key splits: enough waves to fill the chip when the launch has few row tiles, two 32-key chunks a split and more (before the number is rounded up to fours:
// of 576 keys' twelve splits three stay without keys).  Heads of 64 and 128:
// five waves of the step form fill a CU (1024 and 2048 waves: 32 tokens of 1025 - 2047 keys 39.5 and 41.9 us, 128 of 500 - 1500 109
// and 116); portions of 64 rows and more go undivided to the wide form unless they are few and their keys many (one portion behind
// keys, 32 heads on 8 key heads, wide and split: 32 tokens behind 2000 44.8 and 24.9 us, 100 behind 2000 46.4 and 36.4, 100 behind
// none 21 and 23.5, 8 times 16 behind 500 21.4 and 23.9).  Four splits are merged where they are made and take one launch: that many where
// there would be up to seven, or up to eleven on 64 row tiles and more with 2000 keys and fewer (the other launch is 4 us); multiples of four else, no more than four
// a compute unit (us; splits as they were, four, eight: 32 heads of 128 on 8 key heads, tokens of 700 keys: one 9.4 10.6 9.2, eight 13.0 12.1 12.4, 13 15.2 12.5
// 14.4, 16 15.9 13.1 15.5, 24 22.9 16.1 22.5; of 1500 16 24.4 23.5 23.8; of 3000 13 47 44 37, 16 42.9 46.2 42.0, 24 71 58 67; nine of 2100, 15 splits, 16: 24.1 26.9;
// 18 of 1333 - 4000 48 57).
extern "C" int hxm_biased_attention_plan(const hxm_biased_attn_args* args, int32_t max_kv_len, int32_t* n_splits, int64_t* ws_floats) {
  if (!args || !n_splits || !ws_floats) return HX_ERR_NULL;
  const hxm_biased_attn_args& a = *args;
  *n_splits = 1;
  *ws_floats = 0;
  if (a.form == 1 || a.dtype != HX_BF16 || a.max_q_len < 1 || max_kv_len < 1 || a.dim % 8 || a.vdim % 8 || a.dim > 256 || a.vdim > 256 || a.n_seq < 0) return HX_OK;
  if (a.n_seq == 0 || a.kv_heads < 1) return HX_ERR_SHAPE;
  const int64_t rows = (int64_t)a.max_q_len * (a.n_heads / a.kv_heads), tiles = (int64_t)a.n_seq * a.kv_heads * ((rows + 15) / 16);
  if (tiles < 1) return HX_OK;
  int64_t reach = max_kv_len;
  if (a.mask_kind != HXM_MASK_CAUSAL) reach = std::min<int64_t>(reach, (int64_t)a.mask_size + (a.mask_kind == HXM_MASK_WINDOW ? a.max_q_len : 0));
  const bool whole = a.form == 0 && (a.dim == 64 || a.dim == 128) && (a.vdim == 64 || a.vdim == 128) && a.block_size % 16 == 0;
  int64_t ns = std::min({((whole ? 1024 : 2048) + tiles - 1) / tiles, (reach + 31) / 32 / 2, (int64_t)64});
  if (whole && rows >= 64 && (tiles > 256 || reach < 1024)) ns = 1;
  if (whole && ns > 2 && !between_rounds(tiles)) {
    if (ns < 8 || (reach <= 2000 && ns < 12 && tiles >= 64) || (reach <= 512 && ns == 8)) ns = 4;
    else if (tiles > 128) ns = 7;            // (longer keys and just too many row tiles for eight: waves by themselves)
    else ns = std::min((ns + 3) / 4 * 4, 1024 / tiles / 4 * 4);
  }
  if (ns < 2) return HX_OK;
  *n_splits = (int32_t)ns;
  *ws_floats = tiles * ns * 16 * ((a.vdim + 15) / 16 * 16 + 2);
  return HX_OK;
}
