// moe_mix.hip — mixture of experts for the mix library: a softmax router whose choice can carry a bias, the plan that puts
// the (token, choice) pairs in expert-major order, the grouped product Y = act(X W_e^T) over the rows of every expert,
// and the weighted combine with an optional gated shared expert.  Nothing returns to the host between the router and the
// combine: the products are launched for the most rows there can be and find their expert from the plan's segments.
#include <cfloat>
#include <cmath>
#include "mix_rows.h"
#include "tile_product.h"
#include "../../include/hydra_mix.h"

namespace hxm {
int& last_hip_error();
int check_launch();
}  // namespace hxm

namespace {

using namespace hx;

constexpr int kMaxExperts = 1024;
constexpr int kPerLane = kMaxExperts / 64;

// one wave per token, lane l owns experts l, l + 64, ... (PER of them)
template <int PER>
__global__ __launch_bounds__(256) void route_softmax_topk_kernel(const float* __restrict__ logits, int64_t stride,
                                                                 const float* __restrict__ bias, int64_t n_tokens, int E,
                                                                 int top, float scale, float* __restrict__ weights,
                                                                 int32_t* __restrict__ experts, int renorm) {
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= n_tokens) return;
  const float* row = logits + t * stride;
  constexpr int per = PER;
  float s[PER], c[PER];
  float mx = -FLT_MAX;
#pragma unroll
  for (int i = 0; i < per; ++i) {
    const int e = lane + 64 * i;
    s[i] = e < E ? row[e] : -FLT_MAX;
    mx = fmaxf(mx, s[i]);
  }
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < per; ++i) {
    const int e = lane + 64 * i;
    s[i] = e < E ? expf(s[i] - mx) : 0.f;
    sum += s[i];
  }
  sum = wave_sum(sum);
  const float inv = 1.0f / sum;
#pragma unroll
  for (int i = 0; i < per; ++i) {
    const int e = lane + 64 * i;
    s[i] *= inv;
    c[i] = e < E ? s[i] + (bias ? bias[e] : 0.f) : -FLT_MAX;
  }
  float chosen_sum = 0.f, my_w = 0.f;      // lane k keeps the k-th choice
  int my_e = 0;
  for (int k = 0; k < top; ++k) {
    float best = -FLT_MAX;
    int best_e = INT32_MAX;
    float best_s = 0.f;
  #pragma unroll
  for (int i = 0; i < per; ++i) {
      const int e = lane + 64 * i;
      if (e < E && (c[i] > best)) {      // within a lane experts go up: the first of equals is the lower one
        best = c[i];
        best_e = e;
        best_s = s[i];
      }
    }
    for (int off = 32; off > 0; off >>= 1) {
      const float ob = __shfl_xor(best, off, 64);
      const int oe = __shfl_xor(best_e, off, 64);
      const float os = __shfl_xor(best_s, off, 64);
      if (ob > best || (ob == best && oe < best_e)) {
        best = ob;
        best_e = oe;
        best_s = os;
      }
    }
#pragma unroll
    for (int i = 0; i < per; ++i)
      if (lane + 64 * i == best_e) c[i] = -FLT_MAX;      // taken
    chosen_sum += best_s;
    if (lane == k % 64) {      // (top <= 64 is checked by the host)
      my_w = best_s;
      my_e = best_e;
    }
  }
  if (lane < top) {
    weights[t * top + lane] = (renorm ? my_w / (chosen_sum + 1e-20f) : my_w) * scale;
    experts[t * top + lane] = my_e;
  }
}

// A token's choice by one wave: z[i] is the logit of expert lane + 64 i (-inf past the last).  A choice is a maximum over the wave on
// the vector ALU and a ballot for the lowest expert that holds it; the weights are the softmax of the chosen logits.
template <int PER>
__device__ __forceinline__ void choose_top(const float (&z)[PER], int lane, int E, int top, float* __restrict__ weights, int32_t* __restrict__ experts) {
  uint64_t left[PER];         // the experts not chosen yet
#pragma unroll
  for (int i = 0; i < PER; ++i) left[i] = __ballot(lane + 64 * i < E);
  float my_z = 0.f, first = 0.f;      // lane k keeps the k-th choice
  int my_e = 0;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if ((left[i] >> lane) & 1) best = fmaxf(best, z[i]);
    best = row16_max(best);
    const int bits = __builtin_bit_cast(int, best);
    best = fmaxf(fmaxf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(bits, 0)), __builtin_bit_cast(float, __builtin_amdgcn_readlane(bits, 16))),
                 fmaxf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(bits, 32)), __builtin_bit_cast(float, __builtin_amdgcn_readlane(bits, 48))));
    int chosen = -1, fallback = -1;
#pragma unroll
    for (int i = PER - 1; i >= 0; --i) {
      const uint64_t at = __ballot(z[i] == best) & left[i];
      if (at) chosen = 64 * i + __builtin_ctzll(at);
      if (left[i]) fallback = 64 * i + __builtin_ctzll(left[i]);
    }
    if (chosen < 0) chosen = fallback;                        // (logits that are not numbers: still distinct experts)
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (chosen >= 64 * i && chosen < 64 * (i + 1)) left[i] &= ~(1ull << (chosen & 63));
    if (k == 0) first = best;
    if (lane == k) {
      my_z = best;
      my_e = chosen;
    }
  }
  const float ex = lane < top ? expf(my_z - first) : 0.f;
  const float total = wave_sum(ex);
  if (lane < top) {
    weights[lane] = ex / total;
    experts[lane] = my_e;
  }
}

// Router product and choice in one kernel: a workgroup takes 16 tokens; its waves deal the sum over k among themselves, U
// slices of 16 neighbouring k at a time, with float matrix instructions (16 tokens x 16 experts x 4 k: a lane brings four
// neighbouring k of its token's row and of its experts' rows, element e of every lane makes one instruction), their sums meet
// in LDS in a fixed order, and every wave chooses for the tokens whose number is its own (mod waves).
template <int NT, int WAVES>      // experts in tiles of 16
__global__ __launch_bounds__(64 * WAVES) void router_topk_kernel(const float* __restrict__ x, int64_t x_stride, const float* __restrict__ w,
                                                                 const float* __restrict__ bias, int64_t n_tokens, int64_t K, int E, int top,
                                                                 float* __restrict__ weights, int32_t* __restrict__ experts) {
  constexpr int E16 = 16 * NT;
  __shared__ float sums[WAVES][16][E16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int l16 = lane & 15, kq = lane >> 4;
  const int64_t t0 = (int64_t)blockIdx.x * 16;
  const int64_t row = t0 + l16 < n_tokens ? t0 + l16 : n_tokens - 1;
  const float* xr = x + row * x_stride + 4 * kq;
  const float* wr[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int e = 16 * n + l16 < E ? 16 * n + l16 : E - 1;      // (columns past the last expert are not read afterwards)
    wr[n] = w + (int64_t)e * K + 4 * kq;
  }
  f32x4 acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  const f32x4 zero4 = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int U = NT <= 2 ? 4 : NT <= 4 ? 2 : 1;              // slices in flight
  for (int64_t k0 = 16 * U * wave; k0 < K; k0 += 16 * U * WAVES) {
    f32x4 xv[U], wv[U][NT];
#pragma unroll
    for (int s = 0; s < U; ++s) {
      const int64_t k = k0 + 16 * s;
      const bool in = k + 4 * kq < K;
      const int64_t at = in ? k : -(int64_t)(4 * kq);           // (past the end: the row's start, and not used)
      xv[s] = *reinterpret_cast<const f32x4*>(xr + at);
      if (!in) xv[s] = zero4;
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        wv[s][n] = *reinterpret_cast<const f32x4*>(wr[n] + at);
        if (!in) wv[s][n] = zero4;
      }
    }
#pragma unroll
    for (int s = 0; s < U; ++s)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[s][e], wv[s][n][e], acc[n], 0, 0, 0);
  }
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) sums[wave][4 * kq + r][16 * n + l16] = acc[n][r];
  __syncthreads();
  constexpr int PER = (E16 + 63) / 64;
  for (int tt = wave; tt < 16; tt += WAVES) {
    const int64_t t = t0 + tt;
    if (t >= n_tokens) break;
    float z[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = lane + 64 * i;
      z[i] = -INFINITY;
      if (e < E) {
        float s = 0.f;
#pragma unroll
        for (int v = 0; v < WAVES; ++v) s += sums[v][tt][e];
        z[i] = s + (bias ? bias[e] : 0.f);
      }
    }
    choose_top<PER>(z, lane, E, top, weights + t * top, experts + t * top);
  }
}

// The same for few tokens: a workgroup of sixteen waves a token, a wave an expert after the other, its products on the vector ALU.
// The form above puts sixteen tokens on one CU: their matrix products (float, 4 us for 16 experts of 4096) and the rows that pass
// through its one L1 take what the chip's other CUs could share.  4 of 16 experts of 4096: 32 tokens 17.3 us above, 6.7 here; 4 of
// 128: 67 and 33 us.
__global__ __launch_bounds__(1024) void router_few_kernel(const float* __restrict__ x, int64_t x_stride, const float* __restrict__ w,
                                                          const float* __restrict__ bias, int64_t K, int E, int top,
                                                          float* __restrict__ weights, int32_t* __restrict__ experts) {
  __shared__ float logits[128];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t t = blockIdx.x;
  const float* xr = x + t * x_stride;
  for (int e = wave; e < E; e += 16) {
    const float* wr = w + (int64_t)e * K;
    constexpr int U = 8;                                   // pieces of 256 in flight
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int64_t k0 = 4 * lane; k0 < K; k0 += 256 * U) {
      f32x4 xv[U], wv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t k = k0 + 256 * u < K ? k0 + 256 * u : 4 * lane;      // (past the end: the lane's first, and not used)
        xv[u] = *reinterpret_cast<const f32x4*>(xr + k);
        wv[u] = *reinterpret_cast<const f32x4*>(wr + k);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = k0 + 256 * u < K;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = in ? __builtin_fmaf(xv[u][i], wv[u][i], acc[i]) : acc[i];
      }
    }
    const float sum = wave_sum((acc[0] + acc[1]) + (acc[2] + acc[3]));
    if (lane == 0) logits[e] = sum + (bias ? bias[e] : 0.f);
  }
  __syncthreads();
  if (wave > 0) return;
  float z[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) z[i] = lane + 64 * i < E ? logits[lane + 64 * i] : -INFINITY;
  choose_top<2>(z, lane, E, top, weights + t * top, experts + t * top);
}

// Four tokens a workgroup, products on the vector ALU: a wave takes 256 neighbouring k (1 KB of every row) of all four tokens and of NG groups of eight experts, a lane
// sums its k of 32 pairs of a token and an expert, and a transposing sum over the wave leaves one of them in every second lane.
// What bounds the form with sixteen tokens a workgroup is what one CU gets from memory (about 25 bytes a ns: 256 KB of tokens are 10 us), with most CUs idle up to a few
// thousand tokens; here every CU has rows, and the experts' come from its L2 a quarter as often as with a workgroup a token.  Above (or a workgroup a token, *) and
// here, us: 16 experts of 4096, 32 tokens 6.6* 6.2, 400 11.7* 7.0, 1000 17.5 8.3, 2500 18.9 15.5, 4000 23.9 25.2; of 2048, 1000 10.6 6.4; 8 experts of 4096, 4000 22.5
// 18.7; 32 of 4096, 400 18.9* 13.3, 1000 24.8 14.5, 1500 25.0 25.4.
template <int NG, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void router_four_kernel(const float* __restrict__ x, int64_t x_stride, const float* __restrict__ w, const float* __restrict__ bias,
                                                                int64_t n_tokens, int64_t K, int E, int top, float* __restrict__ weights, int32_t* __restrict__ experts) {
  __shared__ float sums[WAVES][4][8 * NG];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t t0 = (int64_t)blockIdx.x * 4;
  float acc[NG][32];
#pragma unroll
  for (int n = 0; n < NG; ++n)
#pragma unroll
    for (int i = 0; i < 32; ++i) acc[n][i] = 0.f;
  for (int64_t k0 = 256 * wave; k0 < K; k0 += 256 * WAVES) {
    const bool in = k0 + 4 * lane < K;
    const int64_t k = in ? k0 + 4 * lane : 0;             // (past the end: the row's start, and not used)
    f32x4 xv[4], wv[NG][8];
#pragma unroll
    for (int t = 0; t < 4; ++t) xv[t] = *reinterpret_cast<const f32x4*>(x + (t0 + t < n_tokens ? t0 + t : n_tokens - 1) * x_stride + k);
#pragma unroll
    for (int n = 0; n < NG; ++n)
#pragma unroll
      for (int e = 0; e < 8; ++e) wv[n][e] = *reinterpret_cast<const f32x4*>(w + (int64_t)(8 * n + e < E ? 8 * n + e : E - 1) * K + k);
    if (!in) {
#pragma unroll
      for (int t = 0; t < 4; ++t) xv[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int n = 0; n < NG; ++n)
#pragma unroll
        for (int e = 0; e < 8; ++e) wv[n][e] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int n = 0; n < NG; ++n)
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int t = 0; t < 4; ++t) acc[n][8 * t + e] = __builtin_fmaf(xv[t][i], wv[n][e][i], acc[n][8 * t + e]);
  }
#pragma unroll
  for (int n = 0; n < NG; ++n) {
    const float sum = transpose_sum32(acc[n], lane);
    if ((lane & 1) == 0) sums[wave][lane >> 4][8 * n + (lane >> 1 & 7)] = sum;
  }
  __syncthreads();
  if (wave >= 4 || t0 + wave >= n_tokens) return;
  float z[1] = {-INFINITY};
  if (lane < E) {
    // (in double: weights' error against 64 bits for 16 experts of 4096 is 1.01e-7 with these added up in float, 0.80 so, 0.97 with a workgroup a token)
    double s = bias ? bias[lane] : 0.f;
#pragma unroll
    for (int v = 0; v < WAVES; ++v) s += sums[v][wave][lane];
    z[0] = (float)s;
  }
  choose_top<1>(z, lane, E, top, weights + (t0 + wave) * top, experts + (t0 + wave) * top);
}

// one workgroup of 1024 threads: histogram, exclusive scan, scatter, all through LDS counters
__global__ __launch_bounds__(1024) void moe_plan_kernel(const int32_t* __restrict__ experts, int64_t n, int top, int E,
                                                        int32_t* __restrict__ seg, int32_t* __restrict__ row_of,
                                                        int32_t* __restrict__ src) {
  __shared__ int32_t count[kMaxExperts];
  __shared__ int32_t cursor[kMaxExperts];
  for (int e = threadIdx.x; e < E; e += 1024) count[e] = 0;
  __syncthreads();
  for (int64_t i = threadIdx.x; i < n; i += 1024) {
    const int e = experts[i];
    if (e >= 0 && e < E) atomicAdd(&count[e], 1);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int32_t run = 0;
    for (int e = 0; e < E; ++e) {
      cursor[e] = run;
      seg[e] = run;
      run += count[e];
    }
    seg[E] = run;
  }
  __syncthreads();
  for (int64_t i = threadIdx.x; i < n; i += 1024) {
    const int e = experts[i];
    if (e >= 0 && e < E) {
      const int32_t row = atomicAdd(&cursor[e], 1);
      row_of[i] = row;
      src[row] = (int32_t)(i / top);
    } else {
      row_of[i] = -1;
    }
  }
}

// the expert and the first row of row tile `tile` (tiles of TM rows, every expert's rows starting a tile of their own);
// false: the tile lies beyond the last expert's rows
__device__ __forceinline__ bool find_tile(const int32_t* __restrict__ seg, int E, int TM, int tile, int& expert, int& row0, int& row1) {
  int passed = 0;
  for (int e = 0; e < E; ++e) {
    const int lo = seg[e], hi = seg[e + 1];
    const int nt = (hi - lo + TM - 1) / TM;
    if (tile < passed + nt) {
      expert = e;
      row0 = lo + (tile - passed) * TM;
      row1 = hi < row0 + TM ? hi : row0 + TM;
      return true;
    }
    passed += nt;
  }
  return false;
}

// The same by the lanes of a wave, an expert each (one expert behind the other is a chain of loads: 1 us with 8 experts, 3 - 4 with 32, in
// launches of 6 - 30): 64 experts from e0 on, their rows, their row tiles and those up to and with them.
struct ExpertTiles {
  int lo, hi, nt, run;
  __device__ __forceinline__ ExpertTiles(const int32_t* __restrict__ seg, int E, int e0, int TM, int lane)
      : lo(seg[min(e0 + lane, E)]), hi(seg[min(e0 + lane + 1, E)]), nt((hi - lo + TM - 1) / TM), run(nt) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int before = __shfl_up(run, d, 64);
      run += lane >= d ? before : 0;
    }
  }
  __device__ __forceinline__ int total() const { return __builtin_amdgcn_readlane(run, 63); }
};

__device__ __forceinline__ float act_apply(float v, int act) {
  if (act == 1) {
    v = fmaxf(v, 0.f);
    return v * v;
  }
  return v;
}

// a clamped gated activation in a product's epilogue (limit <= 0: no clamp)
struct Glu {
  float limit, alpha, up_shift;
  template <typename A>
  __device__ __forceinline__ float of(float g, float u) const {
    if (limit > 0.f) {
      g = fminf(g, limit);
      u = fminf(fmaxf(u, -limit), limit);
    }
    return g * sigmoid_of<A>(alpha * g) * (u + up_shift);
  }
};

// General form (any dtype, any sizes): a workgroup takes 16 rows of one expert and 64 output columns; the rows' inputs go
// through LDS in slices of 64 k; thread (r, c): row r = tid / 16 ... each thread 4 columns.
constexpr int kGM = 16, kGN = 64, kGK = 64;
template <typename A>
__global__ __launch_bounds__(256) void grouped_linear_kernel(typename A::storage* __restrict__ y, const typename A::storage* __restrict__ x,
                                                             int64_t x_stride, const int32_t* __restrict__ src,
                                                             const typename A::storage* __restrict__ w,
                                                             const int32_t* __restrict__ seg, int E, int64_t N, int64_t K, int act, Glu glu) {
  __shared__ float xs[kGM][kGK + 1];
  __shared__ float ws[kGN][kGK + 1];
  int e, row0, row1;
  if (!find_tile(seg, E, kGM, blockIdx.y, e, row0, row1)) return;
  const int64_t col0 = (int64_t)blockIdx.x * kGN;
  const int r = threadIdx.x >> 4, cg = threadIdx.x & 15;      // row r, columns cg, cg + 16, cg + 32, cg + 48
  const typename A::storage* we = w + (int64_t)e * N * K;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int64_t k0 = 0; k0 < K; k0 += kGK) {
    for (int i = threadIdx.x; i < kGM * kGK; i += 256) {
      const int rr = i / kGK, kk = i - rr * kGK;
      float v = 0.f;
      if (row0 + rr < row1 && k0 + kk < K) {
        const int64_t sr = src ? (int64_t)src[row0 + rr] : (int64_t)(row0 + rr);
        v = A::to_float(x[sr * x_stride + k0 + kk]);
      }
      xs[rr][kk] = v;
    }
    for (int i = threadIdx.x; i < kGN * kGK; i += 256) {
      const int cc = i / kGK, kk = i - cc * kGK;
      ws[cc][kk] = (col0 + cc < N && k0 + kk < K) ? A::to_float(we[(col0 + cc) * K + k0 + kk]) : 0.f;
    }
    __syncthreads();
#pragma unroll 8
    for (int kk = 0; kk < kGK; ++kk) {
      const float xv = xs[r][kk];
      acc[0] += xv * ws[cg][kk];
      acc[1] += xv * ws[cg + 16][kk];
      acc[2] += xv * ws[cg + 32][kk];
      acc[3] += xv * ws[cg + 48][kk];
    }
    __syncthreads();
  }
  if (act == 2) {      // columns in turns of 16 gates and 16 ups
    if (row0 + r < row1) {
      for (int j = 0; j < 2; ++j)
        if (col0 + 32 * j < N) y[(int64_t)(row0 + r) * (N >> 1) + (col0 >> 1) + 16 * j + cg] = A::from_float(glu.of<A>(acc[2 * j], acc[2 * j + 1]));
    }
    return;
  }
  if (row0 + r < row1) {
    for (int j = 0; j < 4; ++j) {
      const int64_t c = col0 + cg + 16 * j;
      if (c < N) y[(int64_t)(row0 + r) * N + c] = A::from_float(act_apply(acc[j], act));
    }
  }
}

// MFMA form (bfloat16, K a multiple of 8, rows 16-byte aligned).  A workgroup of WGM x WGN waves takes TM rows of one expert
// and TN output columns.  The rows' inputs (gathered through src) and the expert's weight rows go straight from memory to LDS
// (no registers, no writes by the waves) in slices of 64 k and NS slots; every wave multiplies its (TM / WGM) x (TN / WGN)
// part with 16x16x32 MFMAs: lane l holds k 8 (l / 16) .. + 7 of row (A) or column (B) l % 16, the accumulator's lane l
// column l % 16 of rows 4 (l / 16) .. + 3.  Half a slice is multiplied while the other half's operands are read from LDS, a
// read between two products in tiles of 256 rows, one in those of 128 and of 64 x 128 (narrower tiles have fewer products than reads, in the compiler's order); the one workgroup barrier of a slice stands between its halves, so that a wave always has
// products to issue behind it.
// With few rows an expert it is bound by the weights: those of an expert with one row tile are read past the caches (128 rows of 16
// experts, 2 x 2752 outputs of 4096 and back: 162 + 75 us through registers in tiles of 128 x 128 and padded LDS rows, 115 + 58 us here,
// 6.2 TB/s).  Many rows take grouped_linear_tile_kernel where they can; in tiles of 256 x 256 this form is bound by LDS bandwidth.
// A slice's row is 128 bytes, unpadded (64 lanes land 16 bytes each one after the other): its 16-byte chunk c sits at position
// c ^ (row / 2 % 8), so that the 16 lanes that one pass of a 16-byte LDS read serves — rows 0-3, 12-15 of one k group and
// 4-11 of the next — fall into different banks.
// Workgroups are numbered so that the eight XCDs (dealt round robin) work on eight runs of tiles, the row tiles of an expert
// next to each other: they share the weight columns in the XCD's L2.
constexpr int kKS = 64;
template <int N>
__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

template <int TM, int TN, int WGM, int WGN, int NS, bool FAR>
__global__ __launch_bounds__(64 * WGM * WGN) void grouped_linear_mfma_kernel(u16* __restrict__ y, const u16* __restrict__ x, int64_t x_stride,
                                                                             const int32_t* __restrict__ src, const u16* __restrict__ w,
                                                                             const int32_t* __restrict__ seg, int E, int64_t N, int64_t K,
                                                                             int act, Glu glu) {
  constexpr int NW = WGM * WGN, FM = TM / WGM / 16, FN = TN / WGN / 16;
  constexpr int GA = TM / 8 / NW, GB = TN / 8 / NW;        // load instructions of a wave and slice: eight rows each
  constexpr int kSlice = (TM + TN) * 2 * kKS;              // bytes
  static_assert(GA * NW * 8 == TM && GB * NW * 8 == TN && FN % 2 == 0, "whole groups of eight rows a wave, columns in pairs");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int n_col = (int)((N + TN - 1) / TN);
  int e = 0, row0 = 0, row1 = 0;
  int64_t col0 = 0;
  bool once = false;                                       // the expert has one row tile: nobody reads its weights again
  {
    const int expert_lane = threadIdx.x & 63;
    ExpertTiles some(seg, E, 0, TM, expert_lane);
    int m_tiles = some.total();
    for (int e0 = 64; e0 < E; e0 += 64) m_tiles += ExpertTiles(seg, E, e0, TM, expert_lane).total();
    const int total = m_tiles * n_col, per = (total + 7) >> 3;
    const int at = (int)(blockIdx.x >> 3);
    int tile = (int)(blockIdx.x & 7) * per + at;
    if (at >= per || tile >= total) return;                // (the whole workgroup: no barrier is left waiting)
    for (;;) {
      const uint64_t behind = __builtin_amdgcn_ballot_w64(tile < some.run * n_col);
      if (behind) {
        const int l = __builtin_ctzll(behind), nt = __builtin_amdgcn_readlane(some.nt, l);
        tile -= (__builtin_amdgcn_readlane(some.run, l) - nt) * n_col;
        const int c = tile / nt;
        e += l;
        row0 = __builtin_amdgcn_readlane(some.lo, l) + (tile - c * nt) * TM;
        row1 = min(__builtin_amdgcn_readlane(some.hi, l), row0 + TM);
        col0 = (int64_t)c * TN;
        once = nt == 1;
        break;
      }
      tile -= some.total() * n_col;
      e += 64;
      some = ExpertTiles(seg, E, e, TM, expert_lane);
    }
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm0 = (wave / WGN) * (TM / WGM), wn0 = (wave % WGN) * (TN / WGN);
  const u16* wt = w + ((int64_t)e * N + col0) * K;         // the tile's first weight row
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  // where a lane's 16 bytes of every load come from (a row or column past the last one repeats it; never stored)
  uint32_t oa[GA], ob[GB];
  const u16* pa[GA];
#pragma unroll
  for (int j = 0; j < GA; ++j) {
    const int grp = wave * GA + j, r = min(row0 + 8 * grp + (lane >> 3), row1 - 1);
    const int64_t at = (src ? (int64_t)src[r] : (int64_t)r) * x_stride + 8 * ((lane & 7) ^ (((grp & 1) << 2) + (lane >> 4)));
    if constexpr (FAR) pa[j] = x + at;
    else oa[j] = (uint32_t)(2 * at);
  }
#pragma unroll
  for (int j = 0; j < GB; ++j) {
    const int grp = wave * GB + j;
    const int64_t left = N - 1 - col0;
    const int64_t c = 8 * grp + (lane >> 3) < left ? 8 * grp + (lane >> 3) : left;
    ob[j] = (uint32_t)(2 * (c * K + 8 * ((lane & 7) ^ (((grp & 1) << 2) + (lane >> 4)))));
  }
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  // (m0, the LDS address of the transfer, is a reserved register: nothing else in this kernel uses it)
  auto bring = [&](int64_t k0, int slot) __attribute__((always_inline)) {
    const uint32_t to = lds0 + (uint32_t)(slot * kSlice);
#pragma unroll
    for (int j = 0; j < GA; ++j) {
      const uint32_t at = __builtin_amdgcn_readfirstlane(to + (uint32_t)(wave * GA + j) * 1024u);
      if constexpr (FAR) asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(pa[j] + k0), "s"(at) : "memory", "m0");
      else asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(oa[j]), "s"(x + k0), "s"(at) : "memory", "m0");
    }
    const uint32_t tb = to + (uint32_t)(2 * kKS * TM + wave * GB * 1024);
    if (TM < 256 && once) {
#pragma unroll
      for (int j = 0; j < GB; ++j)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(ob[j]), "s"(wt + k0), "s"(__builtin_amdgcn_readfirstlane(tb + 1024u * j)) : "memory", "m0");
    } else {
#pragma unroll
      for (int j = 0; j < GB; ++j)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(ob[j]), "s"(wt + k0), "s"(__builtin_amdgcn_readfirstlane(tb + 1024u * j)) : "memory", "m0");
    }
  };
#pragma clang diagnostic pop
  const int l16 = lane & 15, kq = lane >> 4;
  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool live = row0 + wm0 < row1;                     // a wave past the expert's rows only helps to bring the slices in
  // a half slice's operands and its products
  struct Frags {
    u16x8 a[FM], b[FN];
  };
  auto read = [&](Frags& f, int slot, int half) __attribute__((always_inline)) {
    const int chunk = ((4 * half + kq) ^ ((l16 >> 1) & 7)) * 16;
    const char* A = smem + slot * kSlice + (wm0 + l16) * 128 + chunk;
    const char* B = smem + slot * kSlice + (TM + wn0 + l16) * 128 + chunk;
#pragma unroll
    for (int j = 0; j < FN; ++j) f.b[j] = *reinterpret_cast<const u16x8*>(B + j * 2048);
#pragma unroll
    for (int i = 0; i < FM; ++i) f.a[i] = *reinterpret_cast<const u16x8*>(A + i * 2048);
  };
  auto multiply = [&](const Frags& f) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, f.a[i]), __builtin_bit_cast(bf16x8, f.b[j]),
                                                            acc[i][j], 0, 0, 0);
  };
  // the reads of one half slice dealt between the products of the other
  auto interleave = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < FM + FN; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, FM * FN / (FM + FN), 0);
    }
  };
  const int n_whole = (int)(K / kKS);
#pragma unroll
  for (int p = 0; p < NS; ++p)
    if (p < n_whole) bring((int64_t)p * kKS, p);
  if (n_whole >= NS) wait_loads<(NS - 1) * (GA + GB)>();
  else wait_loads<0>();
  lds_barrier();
  Frags f0, f1;
  if (n_whole && live) read(f0, 0, 0);
  int slot = 0;
  for (int t = 0; t < n_whole; ++t) {
    const int next = slot == NS - 1 ? 0 : slot + 1;
    if (live) {
      read(f1, slot, 1);
      multiply(f0);
      interleave();
    }
    if (t + 1 < n_whole) {
      // slice t + 1 is there when at most the NS - 2 slices behind it are on their way; past the barrier every wave's part of
      // it is, and every wave has read all of slice t: its slot can be filled again
      if (n_whole - 2 - t >= NS - 2) wait_loads<(NS - 2) * (GA + GB)>();
      else wait_loads<0>();
      lds_barrier();
      if (t + NS < n_whole) bring((int64_t)(t + NS) * kKS, slot);
    }
    if (live) {
      read(f0, next, 0);                                   // (behind the last slice: whatever the slot holds, never used)
      multiply(f1);
      interleave();
    }
    slot = next;
  }
  if (K % kKS) {                                           // the last slice, part of it past K: through registers, zeros there
    const int64_t k0 = (int64_t)n_whole * kKS;
    const u16x8 zero8 = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    __syncthreads();                                       // every wave is done with the slices
#pragma unroll
    for (int j = 0; j < GA; ++j) {
      const int grp = wave * GA + j;
      const bool in = k0 + 8 * ((lane & 7) ^ (((grp & 1) << 2) + (lane >> 4))) < K;
      const char* from;
      if constexpr (FAR) from = reinterpret_cast<const char*>(pa[j] + k0);
      else from = reinterpret_cast<const char*>(x + k0) + oa[j];
      *reinterpret_cast<u16x8*>(smem + grp * 1024 + lane * 16) = in ? *reinterpret_cast<const u16x8*>(from) : zero8;
    }
#pragma unroll
    for (int j = 0; j < GB; ++j) {
      const int grp = wave * GB + j;
      const bool in = k0 + 8 * ((lane & 7) ^ (((grp & 1) << 2) + (lane >> 4))) < K;
      *reinterpret_cast<u16x8*>(smem + 2 * kKS * TM + grp * 1024 + lane * 16) =
          in ? *reinterpret_cast<const u16x8*>(reinterpret_cast<const char*>(wt + k0) + ob[j]) : zero8;
    }
    __syncthreads();
    if (live) {
      read(f0, 0, 0);
      read(f1, 0, 1);
      multiply(f0);
      multiply(f1);
    }
  }
  if (!live) return;
  if (act == 2) {      // columns in turns of 16 gates and 16 ups: a lane holds both numbers of a pair
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; j += 2) {
        const int64_t c = col0 + wn0 + 16 * j;
        if (c >= N) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int rr = row0 + wm0 + 16 * i + 4 * kq + r;
          if (rr < row1) y[(int64_t)rr * (N >> 1) + (c >> 1) + l16] = BF16::from_float(glu.of<BF16>(acc[i][j][r], acc[i][j + 1][r]));
        }
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int64_t c = col0 + wn0 + 16 * j + l16;
      if (c >= N) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int rr = row0 + wm0 + 16 * i + 4 * kq + r;
        if (rr < row1) y[(int64_t)rr * N + c] = BF16::from_float(act_apply(acc[i][j][r], act));
      }
    }
}

template <int TM, int TN, int WGM, int WGN, int NS>
int launch_grouped(u16* y, const u16* x, int64_t x_stride, const int32_t* src, const u16* w, const int32_t* seg, int64_t max_rows, int E,
                   int64_t N, int64_t K, int act, const Glu& glu, hipStream_t s) {
  // every expert's rows start a tile of their own
  const int64_t grid = ((max_rows + TM - 1) / TM + E) * ((N + TN - 1) / TN) + 7;
  if (grid > 0x7fffffff) return HX_ERR_SHAPE;
  constexpr size_t lds = (size_t)NS * (TM + TN) * 2 * kKS;
  // Offsets of 32 bits (bytes) only for rows that come as they are, of which max_rows is the number: src may name any row of x, and how
  // many there are is not known here.
  const bool far = src || max_rows * x_stride > 0x3fffffff;
  auto kernel = far ? grouped_linear_mfma_kernel<TM, TN, WGM, WGN, NS, true> : grouped_linear_mfma_kernel<TM, TN, WGM, WGN, NS, false>;
  if (lds > 64 * 1024) (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  kernel<<<dim3((unsigned)grid), dim3(64 * WGM * WGN), lds, s>>>(y, x, x_stride, src, w, seg, E, N, K, act, glu);
  return hxm::check_launch();
}

// Many rows an expert: tiles of 256 rows and 256 columns (tile_product.h), one workgroup a CU that goes from tile to tile: the
// first slices of the next one are on their way while the results of the last are stored.  Measured with 16 experts, 2 x 2752 outputs
// of 4096 and back: 15956 rows 640 + 373 us in the form above, 585 + 318 us here (1.35 and 1.22 PFLOP/s with what is multiplied
// for rows and columns past the end), where normal data takes all of the card's power.
template <bool FAR>
struct GroupedLoader {
  const u16 *x, *w;               // (at the stream's k)
  uint32_t ox[8], ow[8];          // bytes
  const u16* px[8];
  __device__ __forceinline__ void go(const u16* x_, int64_t x_stride, const int32_t* src, const u16* wt, int64_t K, int row0, int row1, int64_t cols) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    x = x_;
    w = wt;
    // (a row or column past the last one repeats it; never stored)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = min(row0 + tile_load_row(wave, j, lane), row1 - 1);
      const int64_t at = (src ? (int64_t)src[r] : (int64_t)r) * x_stride + tile_load_k(j, lane);
      if constexpr (FAR) px[j] = x_ + at;
      else ox[j] = (uint32_t)(2 * at);
      const int c = tile_load_row(wave, j, lane);
      ow[j] = (uint32_t)(2 * ((c < cols ? c : cols - 1) * K + tile_load_k(j, lane)));
    }
  }
  template <int J>
  __device__ __forceinline__ void a(uint32_t lds) {
    if constexpr (FAR) {
      tile_load<J>(px[J], lds);
      px[J] += kTileK;
    } else {
      tile_load<J>(x, ox[J], lds);
      if constexpr (J == 7) x += kTileK;
    }
  }
  template <int J>
  __device__ __forceinline__ void b(uint32_t lds) {
    tile_load<J>(w, ow[J], lds);
    if constexpr (J == 7) w += kTileK;
  }
};

// K is a multiple of 64 from 128 on, result rows come in whole 16-byte pieces.  GLU: act 2, else 0 or 1.
template <bool FAR, bool GLU>
__global__ __launch_bounds__(256, 1) void grouped_linear_tile_kernel(u16* __restrict__ y, const u16* __restrict__ x, int64_t x_stride,
                                                                     const int32_t* __restrict__ src, const u16* __restrict__ w,
                                                                     const int32_t* __restrict__ seg, int E, int64_t N, int64_t K, int act, Glu glu) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int n_col = (int)((N + kTileRows - 1) / kTileRows), n = (int)(K / kTileK);      // (n >= 2)
  int at, end, e = 0, before = 0;                          // the expert whose tiles are walked, tiles in front of it
  {
    const int expert_lane = threadIdx.x & 63;
    ExpertTiles some(seg, E, 0, kTileRows, expert_lane);
    int m_tiles = some.total();
    for (int e0 = 64; e0 < E; e0 += 64) m_tiles += ExpertTiles(seg, E, e0, kTileRows, expert_lane).total();
    const int total = m_tiles * n_col, per = (total + 7) >> 3;
    at = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    end = min(total, (int)(blockIdx.x & 7) * per + per);
    if (at >= end) return;                                 // (the whole workgroup)
    for (;;) {                                             // the first tile's expert
      const uint64_t behind = __builtin_amdgcn_ballot_w64(at - before < some.run * n_col);
      if (behind) {
        const int l = __builtin_ctzll(behind);
        e += l;
        before += (__builtin_amdgcn_readlane(some.run, l) - __builtin_amdgcn_readlane(some.nt, l)) * n_col;
        break;
      }
      before += some.total() * n_col;
      e += 64;
      some = ExpertTiles(seg, E, e, kTileRows, expert_lane);
    }
  }
  const int step = (int)(gridDim.x >> 3);
  struct Tile {
    int e, row0, row1;
    int64_t col0;
  } tile, next;
  auto find = [&](int i) __attribute__((always_inline)) {
    for (;; ++e) {
      const int r0 = seg[e], r1 = seg[e + 1], nt = (r1 - r0 + kTileRows - 1) / kTileRows, in = i - before;
      if (in < nt * n_col) {
        const int c = in / nt, row0 = r0 + (in - c * nt) * kTileRows;
        return Tile{e, row0, min(r1, row0 + kTileRows), (int64_t)c * kTileRows};
      }
      before += nt * n_col;
    }
  };
  GroupedLoader<FAR> loader;
  auto go = [&](const Tile& t) __attribute__((always_inline)) {
    loader.go(x, x_stride, src, w + ((int64_t)t.e * N + t.col0) * K, K, t.row0, t.row1, N - t.col0);
  };
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm0 = (wave >> 1) * 128, wn0 = (wave & 1) * 128, l16 = lane & 15;
  const int64_t out = GLU ? N >> 1 : N;
  TileProduct<BF16, GroupedLoader<FAR>> p(smem, loader);
  tile = find(at);
  go(tile);
  p.start();
  for (;;) {
    at += step;
    for (int t = 0; t < n; ++t) {
      if (t == n - 2) {                                    // from here on the next tile's slices are requested (behind the last: its own again)
        next = at < end ? find(at) : tile;
        go(next);
      }
      p.slice();
    }
    // a pair of results of 16 columns next to each other, the first at column c of this lane's row r
    auto store = [&](int r, int64_t c, f32x4 first, f32x4 second) __attribute__((always_inline)) {
      const u32x4 v = tile_pair(tile_round<BF16>(first), tile_round<BF16>(second));
      c += tile_pair_column(lane);
      if (r < tile.row1 && c < out) *reinterpret_cast<u32x4*>(y + (int64_t)r * out + c) = v;
    };
    const int64_t c0 = tile.col0 + wn0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = tile.row0 + wm0 + 16 * i + l16;
#pragma unroll
      for (int j = 0; j < 8; j += 4) {
        f32x4 v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = p.take(i, j + q);
        if constexpr (GLU) {      // columns in turns of 16 gates and 16 ups: a lane holds both numbers of a pair
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            v[0][q] = glu.of<BF16>(v[0][q], v[1][q]);
            v[1][q] = glu.of<BF16>(v[2][q], v[3][q]);
          }
          store(r, (c0 >> 1) + 8 * j, v[0], v[1]);
        } else {
#pragma unroll
          for (int q = 0; q < 16; ++q) v[q >> 2][q & 3] = act_apply(v[q >> 2][q & 3], act);
          store(r, c0 + 16 * j, v[0], v[1]);
          store(r, c0 + 16 * j + 32, v[2], v[3]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (at >= end) break;
    tile = next;
    p.clear();
  }
  tile_wait<0>();                                          // (nothing lands in LDS that is no longer this workgroup's)
}

int launch_grouped_tiles(u16* y, const u16* x, int64_t x_stride, const int32_t* src, const u16* w, const int32_t* seg, int64_t max_rows, int E,
                         int64_t N, int64_t K, int act, const Glu& glu, hipStream_t s) {
  const int64_t tiles = ((max_rows + kTileRows - 1) / kTileRows + E) * ((N + kTileRows - 1) / kTileRows);      // every expert's rows start a tile
  if (tiles > 0x7fffffff) return HX_ERR_SHAPE;
  const int64_t grid = tiles < kTileGroups ? (tiles + 7) / 8 * 8 : kTileGroups;      // (the eight XCDs work on a run of tiles each)
  const bool far = src || max_rows * x_stride > 0x3fffffff;
  auto kernel = act == 2 ? (far ? grouped_linear_tile_kernel<true, true> : grouped_linear_tile_kernel<false, true>)
                         : (far ? grouped_linear_tile_kernel<true, false> : grouped_linear_tile_kernel<false, false>);
  (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTileLds);
  kernel<<<dim3((unsigned)grid), dim3(256), kTileLds, s>>>(y, x, x_stride, src, w, seg, E, N, K, act, glu);
  return hxm::check_launch();
}

// A tile's rows and columns.  Up to 32 rows an expert the weights are all there is to read: tiles of 32
// rows and 64 columns.  A slice takes what its bytes need to come from memory, divided by the slices on their way, so tiles are small — few experts
// with rows still are a tile for most compute units — and six slots deep where rows are long; short ones take four, with three workgroups a compute
// unit instead of two (us; 32 x 128 with three slots, 32 x 64 with four, with six: one row, 2 x 704 outputs of 4096 27.5 17.6 16.8 and back 7.5 5.7 5.5;
// 30 rows of 32 such experts 50 45 43 and 24 22 24; 120 rows 68 62 60 and 31 31 34; 2 x 2752 of 4096, 120 rows of 16: 121 117 115 and 62 58 58;
// in the mean of 196 launches of 1 to 256 rows, 8 to 32 experts and depths of 704 to 4096 3 and 2 % above the best of these and four more, 32 x 128 21 %).  More: the form that is expected to take the least
// time, by the rounds of 256 tiles that a compute unit each is given, by the depth of a round and by the weights.  The numbers are fitted (us)
// to 888 launches — 2 to 32 experts, 36 to 450 rows each, drawn evenly, depths of 704 to 5520, 704 to 11040 outputs — with the choices that older measurements over
// 8 to 64 experts had settled kept: 3 % above the best of eleven forms in the mean.  Rows an expert are taken to spread over 0.8 to 1.2 of their mean.
// Eight waves a tile, and tiles of 64 columns besides those of 128: the forms of four waves and 128 columns that stood here took 6 % longer in the mean
// (us, 64 x 64, 64 x 128, 128 x 64, 128 x 128, 256 x 256; those of four waves 64 x 128 and 128 x 128: 8 experts of 2048 x 1408, 57 rows 17 16 14 17 35; 16 18; 16 of
// 1408 x 1024, 100 rows 18 19 17 15 30; 19 16; 8 of 5504 x 4096, 100 rows 113 96 88 99 102; 96 97; 16 of 2048 x 1408, 160 rows 42 35 39 38 40; 38 41; 8 of 1408 x 4096, 256
// rows 64 56 56 44 79; 57 46; 16 of 5504 x 4096, 320 rows 480 384 392 339 289; 386 380).
struct GroupedForm {
  int rows, cols;
  double once, round, depth, weights;        // us; a round; a round and 1024 of depth; a million bytes of weights
};
GroupedForm grouped_form(int64_t max_rows, int E, int64_t N, int64_t K, bool walks) {
  if (max_rows <= (int64_t)32 * E) return GroupedForm{32, 64, 0, 0, 0, 0};
  const GroupedForm forms[5] = {{64, 64, 3.4, 0.86, 3.8, 0.061}, {64, 128, 4.7, 1.4, 5.3, 0.08}, {128, 64, 3.7, 1.5, 7.5, 0.02}, {128, 128, 1.6, 4.4, 10, 0.026},
                                walks ? GroupedForm{256, 256, 4.1, 9.5, 15, 0.11} : GroupedForm{256, 256, 0, 9, 21, 0.08}};
  const double mean = (double)max_rows / E;
  int best = -1;
  double least = 0;
  for (int j = 0; j < 5; ++j) {
    const GroupedForm& f = forms[j];
    double tiles = 0;                         // an expert's
    for (int i = 0; i < 4; ++i) tiles += ceil((0.85 + 0.1 * i) * mean / f.rows) / 4;
    const double full = tiles * E * (double)((N + f.cols - 1) / f.cols) / kTileGroups, rounds = 0.75 * ceil(full) + 0.25 * full;      // (a part of a round takes nearly as long as a whole one)
    const double time = f.once + rounds * (f.round + f.depth * (double)K / 1024) + f.weights * 2e-6 * E * (double)N * (double)K;
    if (best < 0 || time < least) best = j, least = time;
  }
  // Tiles of 192 columns, of 256 by 128 rows, of 192 x 192 instead, where their rounds come out fuller: 8 experts, 66 rows each, 5504 x 4096, are 344 tiles of 128 x 128, two
  // rounds for 256 compute units, and 232 of 128 x 192 (us, 85 and 73); 16 experts, 281 rows, 2816 x 2048 101 and 77 in 192 x 192; 16, 163 rows, 5504 x 4096 197 and 160.
  // Fitted as above, to 2200 launches of 8 to 32 experts whose rows a router with biases deals out (eight points of their spread, the share of a last round that costs as much as a
  // whole one fitted too): 3.6 % less in the mean of them, a tenth or more slower in 52; taken where 8 % less is expected (where any less is: 4 %, and 71).
  if (E < 4 || E > 48) return forms[best];
  struct Fit {
    GroupedForm form;
    double last;
  };
  const Fit fits[8] = {{{64, 64, 4.07, 0, 3.2, 0.0889}, 0.41},      {{64, 128, 3.48, 0.367, 4.9, 0.0942}, 0.657}, {{128, 64, 3.71, 0.666, 5.07, 0.0472}, 0.793}, {{128, 128, 1.65, 3.49, 8.39, 0.0404}, 0.809},
                       {{256, 256, 2.49, 7.95, 19.9, 0.061}, 0.629}, {{128, 192, 1.37, 4.43, 10.7, 0.0574}, 0.77}, {{128, 256, 0.912, 6.68, 13, 0.056}, 0.749},    {{192, 192, 2.1, 5.4, 15.8, 0.0108}, 0.649}};
  auto expected = [&](const Fit& fit) {
    constexpr double spread[8] = {0.72, 0.83, 0.9, 0.97, 1.03, 1.1, 1.17, 1.28};
    const GroupedForm& f = fit.form;
    double tiles = 0;
    for (double q : spread) tiles += ceil(q * mean / f.rows) / 8;
    const double full = tiles * E * (double)((N + f.cols - 1) / f.cols) / kTileGroups, rounds = fit.last * ceil(full) + (1 - fit.last) * full;
    return f.once + rounds * (f.round + f.depth * (double)K / 1024) + f.weights * 2e-6 * E * (double)N * (double)K;
  };
  double limit = 0.92 * expected(fits[best]);
  const GroupedForm* chosen = &forms[best];
  for (int j = 5; j < 8; ++j)
    if (const double time = expected(fits[j]); time < limit) limit = time, chosen = &fits[j].form;
  return *chosen;
}

// The same, NE elements a lane: width, row strides and pointers are multiples of NE elements.  Rows and weights of the
// token's choices are read once into LDS; the choices' rows are requested four at a time, with the shared expert's.  Bound by memory:
// 4 of 16 experts of 4096 and a shared one, 3989 tokens 37.5 us (5.2 TB/s; 42.8 with four elements a lane and a token a workgroup), 2500 tokens of 2048
// 11.8 (14.2).
template <typename A, int NE>
__global__ __launch_bounds__(256) void moe_combine_vec_kernel(typename A::storage* __restrict__ out, const typename A::storage* __restrict__ y,
                                                              const int32_t* __restrict__ row_of, const float* __restrict__ weights,
                                                              const typename A::storage* __restrict__ shared,
                                                              const float* __restrict__ shared_gate, int64_t gate_stride, int top,
                                                              int64_t W, const typename A::storage* __restrict__ identity,
                                                              int64_t identity_stride) {
  __shared__ int32_t rows[64];
  __shared__ float wts[64];
  const int64_t t = blockIdx.x;
  if ((int)threadIdx.x < top) {
    rows[threadIdx.x] = row_of[t * top + threadIdx.x];
    wts[threadIdx.x] = weights[t * top + threadIdx.x];
  }
  __syncthreads();
  const float g = !shared ? 0.f : shared_gate ? 1.0f / (1.0f + expf(-shared_gate[t * gate_stride])) : 1.0f;
  float idw = 0.f;
  if (identity)
    for (int k = 0; k < top; ++k)
      if (rows[k] < 0) idw += wts[k];
  typedef typename A::storage vec __attribute__((ext_vector_type(NE)));
  auto load = [](const typename A::storage* p) { return *reinterpret_cast<const vec*>(p); };
  for (int64_t i = NE * ((int64_t)blockIdx.y * 256 + threadIdx.x); i < W; i += NE * 256 * (int64_t)gridDim.y) {
    float u[NE];
#pragma unroll
    for (int e = 0; e < NE; ++e) u[e] = 0.f;
    vec sh;
    if (shared) sh = load(shared + t * W + i);
    for (int k0 = 0; k0 < top; k0 += 4) {
      vec v[4];
      float w[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const bool there = k0 + k < top && rows[k0 + k < top ? k0 + k : 0] >= 0;
        const int at = there ? k0 + k : 0;
        w[k] = there ? wts[at] : 0.f;
#pragma unroll
        for (int e = 0; e < NE; ++e) v[k][e] = 0;
        if (there) v[k] = load(y + (int64_t)rows[at] * W + i);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int e = 0; e < NE; ++e) u[e] += w[k] * A::to_float(v[k][e]);
    }
    if (idw != 0.f) {
      const vec v = load(identity + t * identity_stride + i);
#pragma unroll
      for (int e = 0; e < NE; ++e) u[e] += idw * A::to_float(v[e]);
    }
    vec o;
#pragma unroll
    for (int e = 0; e < NE; ++e) o[e] = A::from_float(shared ? u[e] + g * A::to_float(sh[e]) : u[e]);
    *reinterpret_cast<vec*>(out + t * W + i) = o;
  }
}

template <typename A>
__global__ __launch_bounds__(256) void moe_combine_kernel(typename A::storage* __restrict__ out, const typename A::storage* __restrict__ y,
                                                          const int32_t* __restrict__ row_of, const float* __restrict__ weights,
                                                          const typename A::storage* __restrict__ shared,
                                                          const float* __restrict__ shared_gate, int64_t gate_stride, int top,
                                                          int64_t W, const typename A::storage* __restrict__ identity,
                                                          int64_t identity_stride) {
  const int64_t t = blockIdx.x;
  const float g = !shared ? 0.f : shared_gate ? 1.0f / (1.0f + expf(-shared_gate[t * gate_stride])) : 1.0f;
  // a choice without a row (an expert past those the plan was made for) is an identity expert when `identity` is given
  float idw = 0.f;
  if (identity)
    for (int k = 0; k < top; ++k)
      if (row_of[t * top + k] < 0) idw += weights[t * top + k];
  for (int64_t i = threadIdx.x; i < W; i += 256) {
    float u = 0.f;
    for (int k = 0; k < top; ++k) {
      const int32_t r = row_of[t * top + k];
      if (r >= 0) u += weights[t * top + k] * A::to_float(y[(int64_t)r * W + i]);
    }
    if (idw != 0.f) u += idw * A::to_float(identity[t * identity_stride + i]);
    if (shared) u += g * A::to_float(shared[t * W + i]);
    out[t * W + i] = A::from_float(u);
  }
}

}  // namespace

extern "C" int hxm_route_softmax_topk(const float* logits, int64_t logit_stride, const float* choice_bias, int64_t n_tokens,
                                      int32_t n_experts, int32_t top, float scale, int32_t renorm, float* weights,
                                      int32_t* experts, void* stream) {
  if (n_tokens < 0 || n_experts < 1 || n_experts > kMaxExperts || top < 1 || top > n_experts || top > 64) return HX_ERR_SHAPE;
  if (n_tokens == 0) return HX_OK;
  if (!logits || !weights || !experts) return HX_ERR_NULL;
  if (logit_stride < n_experts) return HX_ERR_STRIDE;
  const dim3 grid((unsigned)((n_tokens + 3) / 4)), block(256);
  hipStream_t s = (hipStream_t)stream;
#define HXM_ROUTE(PER_) route_softmax_topk_kernel<PER_><<<grid, block, 0, s>>>(logits, logit_stride, choice_bias, n_tokens, \
                                                                              n_experts, top, scale, weights, experts, renorm)
  if (n_experts <= 64) HXM_ROUTE(1);
  else if (n_experts <= 128) HXM_ROUTE(2);
  else if (n_experts <= 256) HXM_ROUTE(4);
  else HXM_ROUTE(kPerLane);
#undef HXM_ROUTE
  return hxm::check_launch();
}

extern "C" int hxm_router_topk(const float* x, int64_t x_stride, const float* w, const float* bias, int64_t n_tokens, int64_t k_dim,
                               int32_t n_experts, int32_t top, float* weights, int32_t* experts, void* stream) {
  if (n_tokens < 0 || k_dim < 4 || k_dim % 4 || n_experts < 1 || n_experts > HXM_ROUTER_MAX_EXPERTS || top < 1 || top > n_experts || top > 64)
    return HX_ERR_SHAPE;
  if (n_tokens == 0) return HX_OK;
  if (!x || !w || !weights || !experts) return HX_ERR_NULL;
  if (x_stride < k_dim || x_stride % 4 || !aligned16(x) || !aligned16(w)) return HX_ERR_STRIDE;
  const dim3 grid((unsigned)((n_tokens + 15) / 16));
  hipStream_t s = (hipStream_t)stream;
  // Four tokens a workgroup: up to 8 experts always, up to 16 and 32 while that reads the experts' rows from L2 less than about 750 and 256 times and the rows are long
  // enough to fill its waves; but a workgroup a token where it is the faster one by a little (us, here and there: 16 experts of 2048, 32 tokens 5.1 4.8, 400 5.4 7.7; 32 of
  // 2048, 128 8.2 7.1, of 1024 6.3 7.1).  Short rows: 16 of 256, 8 tokens 4.0 here and 3.8 below, 2500 5.2 and 4.7; of 512, 1000 4.5 and 5.3; 32 of 512, 8 5.6 and 5.1.
  // Four waves of up to 512 registers are fewer rows in flight than eight, and more workgroups a CU: 16 of 4096, 400 tokens 8.0 and 7.0, 2500 15.5 and 17.8.
  const bool four = n_experts <= 8    ? true
                    : n_experts <= 16 ? (n_tokens <= 1024 ? k_dim >= 512 && (k_dim < 2048 || k_dim >= 4096 || n_tokens > 128) : n_tokens <= 3072 && k_dim >= 1024)
                                      : n_experts <= 32 && n_tokens <= 1024 && k_dim >= 1024 && (k_dim < 2048 || n_tokens > 256);
  if (four) {
    const dim3 fours((unsigned)((n_tokens + 3) / 4));
#define HXM_FOUR(NG_, W_) router_four_kernel<NG_, W_><<<fours, dim3(64 * W_), 0, s>>>(x, x_stride, w, bias, n_tokens, k_dim, n_experts, top, weights, experts)
    if (n_experts <= 8) {
      if (n_tokens <= 1024) HXM_FOUR(1, 8);
      else HXM_FOUR(1, 4);
    } else if (n_experts <= 16) {
      if (n_tokens <= 1024) HXM_FOUR(2, 8);
      else HXM_FOUR(2, 4);
    } else {
      HXM_FOUR(4, 4);
    }
#undef HXM_FOUR
    return hxm::check_launch();
  }
  // A workgroup a token while the CUs take them in one round, two where the form above takes long (above / a workgroup a token:
  // 16 experts of 4096, 256 tokens 17.4 / 7.3 us, 512 17.5 / 11.7, 1024 17.7 / 20.7; 32 of 2048, 512 13.9 / 12.0; 32 of 1024, 256 8.5 /
  // 7.5, 384 8.5 / 11.3; 128 of 1024, 256 21.1 / 20.5, 384 21.6 / 35.1).  Every token reads all experts' rows then, and short rows are
  // soon multiplied there: 128 of 512, 32 tokens 12.8 / 18.1, 32 of 512 5.7 / 6.6, 16 of 512 5.0 / 4.9.
  if (k_dim >= 1024 && n_tokens <= (n_experts <= 32 && k_dim >= 2048 ? 512 : 256)) {
    router_few_kernel<<<dim3((unsigned)n_tokens), dim3(1024), 0, s>>>(x, x_stride, w, bias, k_dim, n_experts, top, weights, experts);
    return hxm::check_launch();
  }
#define HXM_ROUTER(NT_, WAVES_)                                                                                                  \
  router_topk_kernel<NT_, WAVES_><<<grid, dim3(64 * WAVES_), 0, s>>>(x, x_stride, w, bias, n_tokens, k_dim, n_experts, top, weights, experts)
  if (n_experts <= 16) HXM_ROUTER(1, 16);
  else if (n_experts <= 32) HXM_ROUTER(2, 16);
  else if (n_experts <= 64) HXM_ROUTER(4, 16);
  else HXM_ROUTER(8, 8);      // (64 KB of LDS)
#undef HXM_ROUTER
  return hxm::check_launch();
}

extern "C" int hxm_moe_plan(const int32_t* experts, int64_t n_tokens, int32_t top, int32_t n_experts, int32_t* seg,
                            int32_t* row_of, int32_t* src, void* stream) {
  if (n_tokens < 0 || top < 1 || n_experts < 1 || n_experts > kMaxExperts || n_tokens * top > INT32_MAX) return HX_ERR_SHAPE;
  if (!experts || !seg || !row_of || !src) return HX_ERR_NULL;
  moe_plan_kernel<<<dim3(1), dim3(1024), 0, (hipStream_t)stream>>>(experts, n_tokens * top, top, n_experts, seg, row_of, src);
  return hxm::check_launch();
}

extern "C" int hxm_grouped_linear_tile_rows(int64_t max_rows, int32_t n_experts, int64_t n_dim, int64_t k_dim) {
  if (max_rows < 1 || n_experts < 1 || n_dim < 1 || k_dim < 1) return 0;
  return grouped_form(max_rows, n_experts, n_dim, k_dim, k_dim % kTileK == 0 && k_dim >= 2 * kTileK && n_dim % 8 == 0).rows;
}

extern "C" int hxm_grouped_linear(void* y, const void* x, int64_t x_stride, const int32_t* src, const void* w,
                                  const int32_t* seg, int64_t max_rows, int32_t n_experts, int64_t n_dim, int64_t k_dim,
                                  int32_t act, float glu_limit, float glu_alpha, float glu_up_shift, int dtype, void* stream) {
  if (max_rows < 0 || n_experts < 1 || n_experts > kMaxExperts || n_dim < 1 || k_dim < 1 || act < 0 || act > 2 || (act == 2 && n_dim % 32))
    return HX_ERR_SHAPE;
  if (max_rows == 0) return HX_OK;
  if (!y || !x || !w || !seg) return HX_ERR_NULL;
  if (x_stride < k_dim) return HX_ERR_STRIDE;
  const Glu glu{glu_limit, glu_alpha, glu_up_shift};
  hipStream_t s = (hipStream_t)stream;
  if (dtype == HX_BF16 && k_dim % 8 == 0 && k_dim < (1 << 22) && x_stride % 8 == 0 && aligned16(x) && aligned16(w)) {      // (offsets inside a weight tile: 32 bits)
    u16* yy = (u16*)y;
    const u16 *xx = (const u16*)x, *ww = (const u16*)w;
    const bool walks = k_dim % kTileK == 0 && k_dim >= 2 * kTileK && (act == 2 || n_dim % 8 == 0) && aligned16(y);
    const GroupedForm f = grouped_form(max_rows, n_experts, n_dim, k_dim, walks);
    auto go = [&](auto launch) { return launch(yy, xx, x_stride, src, ww, seg, max_rows, n_experts, n_dim, k_dim, act, glu, s); };
    if (f.rows == 32) return k_dim < 2048 ? go(launch_grouped<32, 64, 2, 2, 4>) : go(launch_grouped<32, 64, 2, 2, 6>);
    if (f.rows == 64) return f.cols == 64 ? go(launch_grouped<64, 64, 4, 2, 3>) : go(launch_grouped<64, 128, 2, 4, 3>);
    if (f.rows == 192) return go(launch_grouped<192, 192, 4, 2, 3>);
    if (f.rows == 128 && f.cols == 192) return go(launch_grouped<128, 192, 4, 2, 3>);
    if (f.rows == 128 && f.cols == 256) return go(launch_grouped<128, 256, 2, 4, 3>);
    if (f.rows == 128) return f.cols == 64 ? go(launch_grouped<128, 64, 4, 2, 3>) : go(launch_grouped<128, 128, 2, 4, 3>);
    return walks ? go(launch_grouped_tiles) : go(launch_grouped<256, 256, 2, 4, 2>);
  }
  const int64_t tiles = (max_rows + kGM - 1) / kGM + n_experts;
  if (tiles > 65535) return HX_ERR_SHAPE;
  const dim3 grid((unsigned)((n_dim + kGN - 1) / kGN), (unsigned)tiles), block(256);
  switch (dtype) {
    case HX_F32:
      grouped_linear_kernel<F32><<<grid, block, 0, s>>>((float*)y, (const float*)x, x_stride, src, (const float*)w, seg, n_experts,
                                                        n_dim, k_dim, act, glu);
      break;
    case HX_BF16:
      grouped_linear_kernel<BF16><<<grid, block, 0, s>>>((u16*)y, (const u16*)x, x_stride, src, (const u16*)w, seg, n_experts, n_dim,
                                                         k_dim, act, glu);
      break;
    default: return HX_ERR_DTYPE;
  }
  return hxm::check_launch();
}

extern "C" int hxm_moe_combine(void* out, const void* y, const int32_t* row_of, const float* weights, const void* shared,
                               const float* shared_gate, int64_t gate_stride, const void* identity, int64_t identity_stride,
                               int64_t n_tokens, int32_t top, int64_t width, int dtype, void* stream) {
  if (n_tokens < 0 || top < 1 || width < 1) return HX_ERR_SHAPE;
  if (identity && identity_stride < width) return HX_ERR_STRIDE;
  if (n_tokens == 0) return HX_OK;
  if (!out || !y || !row_of || !weights) return HX_ERR_NULL;
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)n_tokens), block(256);
  const uintptr_t es = dtype == HX_F32 ? 4 : 2;
  auto by = [&](int ne) {
    auto aligned = [&](const void* p) { return (uintptr_t)p % (ne * es) == 0; };
    return top <= 64 && width % ne == 0 && identity_stride % ne == 0 && aligned(out) && aligned(y) && aligned(shared) && aligned(identity);
  };
  auto vgrid = [&](int ne) {              // a piece of the row a workgroup
    const int64_t pieces = (width + 256 * ne - 1) / (256 * ne);
    return dim3((unsigned)n_tokens, (unsigned)(pieces < 64 ? pieces : 64));
  };
  if (dtype == HX_F32 && by(4)) {
    moe_combine_vec_kernel<F32, 4><<<vgrid(4), block, 0, s>>>((float*)out, (const float*)y, row_of, weights, (const float*)shared, shared_gate, gate_stride, top,
                                                              width, (const float*)identity, identity_stride);
    return hxm::check_launch();
  }
  if (dtype == HX_BF16 && by(4)) {
    const int ne = n_tokens > 256 && by(8) ? 8 : 4;      // (few tokens: more workgroups; 200 tokens of 2048 3.9 and 4.3 us)
    auto kernel = ne == 8 ? moe_combine_vec_kernel<BF16, 8> : moe_combine_vec_kernel<BF16, 4>;
    kernel<<<vgrid(ne), block, 0, s>>>((u16*)out, (const u16*)y, row_of, weights, (const u16*)shared, shared_gate, gate_stride, top, width,
                                                  (const u16*)identity, identity_stride);
    return hxm::check_launch();
  }
  switch (dtype) {
    case HX_F32:
      moe_combine_kernel<F32><<<grid, block, 0, s>>>((float*)out, (const float*)y, row_of, weights, (const float*)shared, shared_gate,
                                                     gate_stride, top, width, (const float*)identity, identity_stride);
      break;
    case HX_BF16:
      moe_combine_kernel<BF16><<<grid, block, 0, s>>>((u16*)out, (const u16*)y, row_of, weights, (const u16*)shared, shared_gate,
                                                      gate_stride, top, width, (const u16*)identity, identity_stride);
      break;
    default: return HX_ERR_DTYPE;
  }
  return hxm::check_launch();
}
