// gemm_rows.hip — the linear layers of batches of prompts (replaces torch.nn.Linear of hydrainfer/model/model_forward.py:36 and
// hydrainfer/layer/causal_attention.py for 65 to about a thousand rows): Y = X W^T in tiles of 64 x 64 to 192 x 192, the depth in up to eight splits whose float
// slabs the add and norm behind the product sum (hx_add_rms_norm_slabs), or gate and up with silu(gate) * up in one launch.
// What bounds such products is tiles enough for 256 compute units and a depth short enough for each: 128 rows of 4096 outputs of 11008 are 32 tiles of 128 x 128
// in the library's way (59.8 us with the add and norm), 256 here with eight splits (29.2 us, 4.2 TB/s of weights and slabs).  A workgroup multiplies one tile: slices of 64 k come straight to
// LDS (no registers, no writes by the waves) in three slots (four in the smallest tiles), half a slice is multiplied while the other half's operands are read, and the one barrier a slice stands between its
// halves.  Products are made as W X^T, so that a lane holds four columns of a row and stores them together.
#include <cmath>

#include "tile_product.h"

namespace hx {
namespace {

constexpr int kSlice = 64;                                 // k of a slice
template <int N>
__device__ __forceinline__ void rows_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ float rows_silu(float x) { return x / (1.0f + __expf(-x)); }

template <typename T, int TM, int TN, int WGM, int WGN, int NS>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm_rows_kernel(u16* __restrict__ out, float* __restrict__ slabs, const u16* __restrict__ x, const u16* __restrict__ w, int M, int N, int K,
                                                                  int ldx, int ldw, int splits, int inter) {
  constexpr int NW = WGM * WGN, FM = TM / WGM / 16, FN = TN / WGN / 16;
  constexpr int GA = TM / 8 / NW, GB = TN / 8 / NW;        // load instructions of a wave and slice: eight rows each
  constexpr int kBytes = (TM + TN) * 2 * kSlice;
  static_assert(GA * NW * 8 == TM && GB * NW * 8 == TN && FN % 2 == 0, "whole groups of eight rows a wave, columns in pairs");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int n_row = (M + TM - 1) / TM, n_col = (N + TN - 1) / TN, total = n_row * n_col * splits, per = (total + 7) >> 3;
  const int at = (int)(blockIdx.x >> 3);
  const int unit = (int)(blockIdx.x & 7) * per + at;
  if (at >= per || unit >= total) return;                  // (the whole workgroup)
  const int row0 = unit % n_row * TM, col0 = unit / n_row % n_col * TN, split = unit / n_row / n_col;
  const int slices = K / kSlice, first = (int)((int64_t)slices * split / splits), n = (int)((int64_t)slices * (split + 1) / splits) - first;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm0 = (wave / WGN) * (TM / WGM), wn0 = (wave % WGN) * (TN / WGN);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  // where a lane's 16 bytes of every load come from (a row or column past the last one repeats it; never stored)
  uint32_t oa[GA], ob[GB];
#pragma unroll
  for (int j = 0; j < GA; ++j) {
    const int grp = wave * GA + j, r = min(row0 + 8 * grp + (lane >> 3), M - 1);
    oa[j] = (uint32_t)(2 * ((int64_t)r * ldx + 8 * ((lane & 7) ^ (((grp & 1) << 2) + (lane >> 4)))));
  }
#pragma unroll
  for (int j = 0; j < GB; ++j) {
    const int grp = wave * GB + j, c = min(col0 + 8 * grp + (lane >> 3), N - 1);
    const int row = inter ? (c >> 5) * 16 + (c & 15) + (c & 16 ? inter : 0) : c;      // (gates and ups in turns of sixteen)
    ob[j] = (uint32_t)(2 * ((int64_t)row * ldw + 8 * ((lane & 7) ^ (((grp & 1) << 2) + (lane >> 4)))));
  }
  x += (int64_t)first * kSlice;
  w += (int64_t)first * kSlice;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  // (m0, the LDS address of the transfer, is a reserved register: nothing else in this kernel uses it)
  auto bring = [&](int t, int slot) __attribute__((always_inline)) {
    const uint32_t to = lds0 + (uint32_t)(slot * kBytes);
#pragma unroll
    for (int j = 0; j < GA; ++j)
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(oa[j]), "s"(x + t * kSlice), "s"(__builtin_amdgcn_readfirstlane(to + (uint32_t)(wave * GA + j) * 1024u)) : "memory", "m0");
    const uint32_t tb = to + (uint32_t)(2 * kSlice * TM + wave * GB * 1024);
#pragma unroll
    for (int j = 0; j < GB; ++j)
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(ob[j]), "s"(w + t * kSlice), "s"(__builtin_amdgcn_readfirstlane(tb + 1024u * j)) : "memory", "m0");
  };
#pragma clang diagnostic pop
  const int l16 = lane & 15, kq = lane >> 4;
  f32x4 acc[FM][FN];                                       // lane l: columns 4 (l / 16) .. + 3 of row l % 16
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Frags {
    u16x8 a[FM], b[FN];
  };
  auto read = [&](Frags& f, int slot, int half) __attribute__((always_inline)) {
    const int chunk = ((4 * half + kq) ^ ((l16 >> 1) & 7)) * 16;
    const char* A = smem + slot * kBytes + (wm0 + l16) * 128 + chunk;
    const char* B = smem + slot * kBytes + (TM + wn0 + l16) * 128 + chunk;
#pragma unroll
    for (int j = 0; j < FN; ++j) f.b[j] = *reinterpret_cast<const u16x8*>(B + j * 2048);
#pragma unroll
    for (int i = 0; i < FM; ++i) f.a[i] = *reinterpret_cast<const u16x8*>(A + i * 2048);
  };
  auto multiply = [&](const Frags& f) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = Mfma<T>::mma(f.b[j], f.a[i], acc[i][j]);
  };
  // the reads of one half slice dealt between the products of the other
  auto interleave = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < FM + FN; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, FM * FN / (FM + FN), 0);
    }
  };
  auto barrier = [&]() __attribute__((always_inline)) {     // orders LDS traffic only: loads stay in flight
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  const bool live = row0 + wm0 < M;                        // a wave past the last row only helps to bring the slices in
#pragma unroll
  for (int p = 0; p < NS; ++p)
    if (p < n) bring(p, p);
  if (n >= NS) rows_wait<(NS - 1) * (GA + GB)>();
  else rows_wait<0>();
  barrier();
  Frags f0, f1;
  if (n && live) read(f0, 0, 0);
  int slot = 0;
  for (int t = 0; t < n; ++t) {
    const int next = slot == NS - 1 ? 0 : slot + 1;
    if (live) {
      read(f1, slot, 1);
      multiply(f0);
      interleave();
    }
    if (t + 1 < n) {
      // slice t + 1 is there when at most the NS - 2 slices behind it are on their way; past the barrier every wave's part of
      // it is, and every wave has read all of slice t: its slot can be filled again
      if (n - 2 - t >= NS - 2) rows_wait<(NS - 2) * (GA + GB)>();
      else rows_wait<0>();
      barrier();
      if (t + NS < n) bring(t + NS, slot);
    }
    if (live) {
      read(f0, next, 0);                                   // (behind the last slice: whatever the slot holds, never used)
      multiply(f1);
      interleave();
    }
    slot = next;
  }
  if (!live) return;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int r = row0 + wm0 + 16 * i + l16;
    if (r >= M) continue;
    if (slabs) {
      float* to = slabs + ((int64_t)split * M + r) * N;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int c = col0 + wn0 + 16 * j + 4 * kq;
        if (c < N) *reinterpret_cast<f32x4*>(to + c) = acc[i][j];
      }
    } else if (inter) {                                    // rounded where the separate launches round
#pragma unroll
      for (int j = 0; j < FN; j += 2) {
        const int c = col0 + wn0 + 16 * j;
        f32x4 v;
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = round_to<T>(rows_silu(round_to<T>(acc[i][j][q]))) * round_to<T>(acc[i][j + 1][q]);
        if (c < N) *reinterpret_cast<u32x2*>(out + (int64_t)r * inter + (c >> 1) + 4 * kq) = tile_round<T>(v);
      }
    } else {
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int c = col0 + wn0 + 16 * j + 4 * kq;
        if (c < N) *reinterpret_cast<u32x2*>(out + (int64_t)r * N + c) = tile_round<T>(acc[i][j]);
      }
    }
  }
}

struct RowsArgs {
  u16* out;
  float* slabs;
  const u16 *x, *w;
  int M, N, K, ldx, ldw, splits, inter;
};
template <typename T, int TM, int TN, int WGM, int WGN, int NS>
int launch_rows(const RowsArgs& a, hipStream_t s) {
  const int64_t units = (int64_t)((a.M + TM - 1) / TM) * ((a.N + TN - 1) / TN) * a.splits;
  constexpr size_t lds = (size_t)NS * (TM + TN) * 2 * kSlice;
  auto kernel = gemm_rows_kernel<T, TM, TN, WGM, WGN, NS>;
  if (lds > 64 * 1024) {
    const int rc = hip_rc(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    if (rc != HX_OK) return rc;
  }
  hx::launcher(kernel, dim3((unsigned)((units + 7) / 8 * 8)), dim3(64 * WGM * WGN), lds, s)(a.out, a.slabs, a.x, a.w, a.M, a.N, a.K, a.ldx, a.ldw, a.splits, a.inter);
  return check_launch();
}
template <typename T>
int launch_form(int form, const RowsArgs& a, hipStream_t s) {
  switch (form) {
    case 0: return launch_rows<T, 64, 64, 4, 2, 4>(a, s);
    case 1: return launch_rows<T, 64, 128, 2, 4, 3>(a, s);
    case 2: return launch_rows<T, 128, 64, 4, 2, 3>(a, s);
    case 3: return launch_rows<T, 128, 128, 2, 4, 3>(a, s);
    case 4: return launch_rows<T, 128, 192, 4, 2, 3>(a, s);
    case 5: return launch_rows<T, 192, 192, 4, 2, 3>(a, s);
    case 6: return launch_rows<T, 128, 256, 2, 4, 3>(a, s);
    case 7: return launch_rows<T, 192, 128, 4, 2, 3>(a, s);
  }
  return HX_ERR_UNSUPPORTED;
}

// The tiles and the splits of k that are expected to take the least time: by rounds of 256 tiles (a compute unit each; last: the share of a part of a round that costs as much as
// a whole one), the depth of a round, the weights, and the slabs that are written and read again.  Fitted (us, with the add and the norm behind them) to 66 to 1300
// rows of widths 2048, 4096 and 5120 in 4800 launches: 1 % above the best of these forms in the mean.
struct RowsFit {
  int rows, cols;
  double once, round, depth, weights, last, slabs;
};
constexpr RowsFit kFits[8] = {{64, 64, 7.08, 0, 3.06, 0.0378, 0.979, 0.184},
                         {64, 128, 7.43, 0, 4.84, 0.0603, 0.717, 0.129},
                         {128, 64, 7.44, 0, 4.73, 0.0546, 0.73, 0.124},
                         {128, 128, 6.69, 0.591, 8.13, 0.0441, 0.822, 0.17},
                         {128, 192, 7.5, 0, 10.9, 0.0396, 0.84, 0.178},
                         {192, 192, 7.86, 0, 14.9, 0.00495, 0.735, 0.182},
                         {128, 256, 6.84, 2.12, 13.4, 0.0371, 0.853, 0.146},
                         {192, 128, 6.81, 0, 11.2, 0.00561, 0.76, 0.198}};
struct RowsPlan {
  int form, splits;
};
RowsPlan rows_plan(int64_t M, int64_t N, int64_t K, bool may_split) {
  RowsPlan plan{0, 1};
  double least = 0;
  for (int f = 0; f < 8; ++f)
    for (int splits : {1, 2, 3, 4, 6, 8}) {
      const RowsFit& t = kFits[f];
      const double units = (double)((M + t.rows - 1) / t.rows) * (double)((N + t.cols - 1) / t.cols) * splits;
      if (splits > 1 && (!may_split || units > 1100 || K / kSlice / splits < 8)) continue;
      const double full = units / 256, rounds = t.last * ceil(full) + (1 - t.last) * full, slabs = may_split ? (splits > 1 ? splits : 0.5) * (double)M * (double)N * 8e-6 : 0;
      const double time = t.once + rounds * (t.round + t.depth * (double)K / 1024 / splits) + t.weights * 2e-6 * (double)N * (double)K + t.slabs * slabs;
      if ((f == 0 && splits == 1) || time < least) plan = RowsPlan{f, splits}, least = time;
    }
  return plan;
}

// (32-bit byte offsets of rows and weight rows, 32-bit counts)
bool rows_fit(int64_t M, int64_t N, int64_t K) { return M >= 1 && N >= 16 && N % 16 == 0 && K >= kSlice && K % kSlice == 0 && M <= (1 << 20) && N <= (1 << 20) && K <= (1 << 20); }
int rows_refusal(const void* x, const void* w, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int dtype) {
  if (!x || !w) return HX_ERR_NULL;
  if (dtype != HX_F16 && dtype != HX_BF16) return HX_ERR_DTYPE;
  if (ldx < K || ldw < K || ldx % 8 || ldw % 8 || !aligned16(x) || !aligned16(w) || ldx > 0x7fffffff / M || ldw > 0x7fffffff / N) return HX_ERR_STRIDE;
  return HX_OK;
}

}  // namespace
}  // namespace hx

using namespace hx;

namespace hx {
// gate and up of fewer rows (gemm_tile.hip's entry sends them here): served and the fastest form
bool gate_up_in_small_tiles(int64_t M, int64_t inter, int64_t K) {
  // Library product and silu_and_mul, one workgroup a CU in tiles of 256 (gemm_tile.hip), and here, us: 2 x 5632 of 2048, 100 rows 19.0 43 14.8, 350 31.5 43 25.9,
  // 600 36.6 45.7 32.6; 2 x 11008 of 4096, 200 64.7 83 55.7, 300 82 84 70, 512 103 101 111; 2 x 13824 of 5120, 200 92 107 86, 300 104 115 115.
  return M > 64 && M <= 1024 && inter % 16 == 0 && rows_fit(M, 2 * inter, K) && M * inter <= 3500000;
}
int gate_up_small_tiles(void* out, const void* x, const void* weight, int64_t M, int64_t inter, int64_t K, int64_t ldx, int64_t ldw, int dtype, hipStream_t s) {
  const RowsArgs a{(u16*)out, nullptr, (const u16*)x, (const u16*)weight, (int)M, (int)(2 * inter), (int)K, (int)ldx, (int)ldw, 1, (int)inter};
  const int form = rows_plan(M, 2 * inter, K, false).form;
  return dtype == HX_F16 ? launch_form<F16>(form, a, s) : launch_form<BF16>(form, a, s);
}
}  // namespace hx

extern "C" int hx_linear_rows_splits(int64_t M, int64_t N, int64_t K) {
  // Where the library's product and add_rms_norm take longer, us, theirs and these with their slabs' sum in the norm: 2048 of 5632, 100 rows 17.5 and 14.0, 350 24.7 22.9, 1000
  // 39.1 35.2, 1700 51.5 53.1; 4096 of 11008, 128 59.8 29.2, 350 62.4 47.3, 1000 114.7 91.2, 2200 170 190; 4096 of 4096, 128 24.3 16.1, 350 27.1 26.4,
  // 600 35.4 36.0; 5120 of 5120, 256 55 30, 600 48.9 49.6.  (More: the library's tiles fill the chip, and are the faster ones.)
  if (M <= 64 || !rows_fit(M, N, K) || N % 32 || M > (K >= 2 * N ? 1024 : 512)) return 0;
  return rows_plan(M, N, K, true).splits;
}

extern "C" int hx_linear_rows(void* out, float* slabs, int32_t n_splits, const void* x, const void* weight, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int dtype,
                              hx_stream stream) {
  if (M < 0 || (M > 0 && (!rows_fit(M, N, K) || N % 32))) return HX_ERR_SHAPE;
  if (M == 0) return HX_OK;
  if (const int rc = rows_refusal(x, weight, M, N, K, ldx, ldw, dtype)) return rc;
  const RowsPlan plan = rows_plan(M, N, K, true);
  if (n_splits != plan.splits) return HX_ERR_SHAPE;
  void* to = plan.splits > 1 ? (void*)slabs : out;
  if (!to) return HX_ERR_NULL;
  if (!aligned16(to)) return HX_ERR_STRIDE;
  const RowsArgs a{(u16*)out, plan.splits > 1 ? slabs : nullptr, (const u16*)x, (const u16*)weight, (int)M, (int)N, (int)K, (int)ldx, (int)ldw, plan.splits, 0};
  return dtype == HX_F16 ? launch_form<F16>(plan.form, a, (hipStream_t)stream) : launch_form<BF16>(plan.form, a, (hipStream_t)stream);
}

extern "C" int hx_linear_rows_whole_supported(int64_t M, int64_t N, int64_t K) {
  // On the GPU these and the library's product take the same time up to K = 2048, us, here and there: 6144 of 2048, 104 rows 12.3 14.0, 256 17.6 23.9, 300 18.2 17.2, 600 22.3
  // 24.5, 1024 29.3 29.6; 4096 of 2048, 160 11.8 16.4, 384 17.1 14.9, 900 21.0 23.7 (0.95 in the mean of 26).  The library's call costs its caller 15 us more, and batches of
  // prompts through layers of that width are bound by their caller up to some 500 tokens.  Deeper products are the library's: 12288 of 4096 104 32.8 29.6, 1024 109 84.
  return M > 64 && M <= 1024 && rows_fit(M, N, K) && N % 32 == 0 && K <= 2048 && N * K <= 6144 * 2048;
}

extern "C" int hx_linear_rows_whole(void* out, const void* x, const void* weight, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int dtype, hx_stream stream) {
  if (M < 0 || (M > 0 && (!rows_fit(M, N, K) || N % 32))) return HX_ERR_SHAPE;
  if (M == 0) return HX_OK;
  if (!out) return HX_ERR_NULL;
  if (const int rc = rows_refusal(x, weight, M, N, K, ldx, ldw, dtype)) return rc;
  if (!aligned16(out)) return HX_ERR_STRIDE;
  const RowsArgs a{(u16*)out, nullptr, (const u16*)x, (const u16*)weight, (int)M, (int)N, (int)K, (int)ldx, (int)ldw, 1, 0};
  const int form = rows_plan(M, N, K, false).form;
  return dtype == HX_F16 ? launch_form<F16>(form, a, (hipStream_t)stream) : launch_form<BF16>(form, a, (hipStream_t)stream);
}
