// gemm_tile.hip — gate and up projection of many rows with silu(gate) * up in the same launch (replaces two of the torch.nn.Linear
// and the activation of hydrainfer/model/model_forward.py:36 for batches of prompts): tiles of 256 rows and 128 + 128 columns by
// tile_product.h, one workgroup a CU that goes from tile to tile.  A tile takes gate rows and up rows of the weight in turns of
// sixteen, so that a lane holds both numbers of a pair; the [rows, 2 inter] product, which is written and read again otherwise, never
// leaves the registers.
// Bound by the card's power with normal data (tile_product.h).  2693 rows, 2 x 11008 outputs of 4096: the library's product 487 us and
// silu_and_mul 28, here 372 (1.31 PFLOP/s).
#include "tile_product.h"

namespace hx {
namespace {

struct GateUpLoader {
  const u16 *x, *w;               // (at the stream's k)
  uint32_t ox[8], ow[8];          // bytes
  template <int J>
  __device__ __forceinline__ void a(uint32_t lds) {
    tile_load<J>(x, ox[J], lds);
    if constexpr (J == 7) x += kTileK;
  }
  template <int J>
  __device__ __forceinline__ void b(uint32_t lds) {
    tile_load<J>(w, ow[J], lds);
    if constexpr (J == 7) w += kTileK;
  }
};

__device__ __forceinline__ float silu_f32(float x) { return x / (1.0f + __expf(-x)); }

// Rows in panels of panel_rows tiles, a panel's columns one after the other, its row tiles next to each other: the eight XCDs (dealt
// round robin) work on a run of tiles each, about as many rows as columns of them at a time.
template <typename T>
__global__ __launch_bounds__(256, 1) void gate_up_silu_rows_kernel(u16* __restrict__ out, const u16* __restrict__ x, const u16* __restrict__ w,
                                                                   int M, int inter, int K, int64_t ldx, int64_t ldw, int panel_rows) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int n_row = (M + kTileRows - 1) / kTileRows, n_col = (inter + kTileRows / 2 - 1) / (kTileRows / 2), n = K / kTileK;
  const int total = n_row * n_col, per = (total + 7) >> 3;
  int at = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  const int end = min(total, (int)(blockIdx.x & 7) * per + per), step = (int)(gridDim.x >> 3);
  if (at >= end) return;                                   // (the whole workgroup)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  GateUpLoader loader;
  int row0, col0;                                          // of the tile whose slices are requested
  auto go = [&](int i) __attribute__((always_inline)) {
    const int panel = i / (panel_rows * n_col), in = i - panel * panel_rows * n_col;
    const int rows = min(panel_rows, n_row - panel * panel_rows), c = in / rows;
    row0 = (panel * panel_rows + in - c * rows) * kTileRows;
    col0 = c * (kTileRows / 2);
    loader.x = x;
    loader.w = w;
    // (a row or column past the last one repeats it; never stored)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int at = tile_load_row(wave, j, lane), r = min(row0 + at, M - 1), o = min(col0 + (at >> 5) * 16 + (at & 15), inter - 1);
      loader.ox[j] = (uint32_t)(2 * (r * ldx + tile_load_k(j, lane)));
      loader.ow[j] = (uint32_t)(2 * ((o + (at & 16 ? inter : 0)) * ldw + tile_load_k(j, lane)));
    }
  };
  TileProduct<T, GateUpLoader> p(smem, loader);
  go(at);
  p.start();
  for (;;) {
    const int r0 = row0 + (wave >> 1) * 128 + (lane & 15), c0 = col0 + (wave & 1) * 64 + tile_pair_column(lane);
    const int now = at;
    at += step;
    for (int t = 0; t < n; ++t) {
      if (t == n - 2) go(at < end ? at : now);             // from here on the next tile's slices (behind the last: its own again)
      p.slice();
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 8; j += 4) {
        f32x4 v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = p.take(i, j + q);
        // (rounded where the separate launches round)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          v[0][q] = round_to<T>(silu_f32(round_to<T>(v[0][q]))) * round_to<T>(v[1][q]);
          v[1][q] = round_to<T>(silu_f32(round_to<T>(v[2][q]))) * round_to<T>(v[3][q]);
        }
        const u32x4 o = tile_pair(tile_round<T>(v[0]), tile_round<T>(v[1]));
        if (r0 + 16 * i < M && c0 + 8 * j < inter) *reinterpret_cast<u32x4*>(out + (int64_t)(r0 + 16 * i) * inter + c0 + 8 * j) = o;
        __builtin_amdgcn_sched_barrier(0);
      }
    if (at >= end) break;
    p.clear();
  }
  tile_wait<0>();                                          // (nothing lands in LDS that is no longer this workgroup's)
}

}  // namespace
}  // namespace hx

namespace hx {
bool gate_up_in_small_tiles(int64_t M, int64_t inter, int64_t K);      // gemm_rows.hip
int gate_up_small_tiles(void* out, const void* x, const void* weight, int64_t M, int64_t inter, int64_t K, int64_t ldx, int64_t ldw, int dtype, hipStream_t s);
}  // namespace hx

using namespace hx;

extern "C" int hx_gate_up_silu_few_rows_supported(int64_t M, int64_t inter, int64_t K) { return gate_up_in_small_tiles(M, inter, K) ? 1 : 0; }

extern "C" int hx_gate_up_silu_rows_supported(int64_t M, int64_t inter, int64_t K) {
  if (M < 1 || inter < 16 || inter % 16 || K < 2 * kTileK || K % kTileK || M > (1 << 24) || inter > (1 << 24) || K > (1 << 24)) return 0;
  // Worth it where at least 0.6 of the rounds of tiles is rows and columns.  Library and silu / here, us: 2 x 11008 outputs of 4096,
  // 600 rows (0.39) 130 / 160, 900 (0.59) 168 / 168, 1300 (0.57) 303 / 247, 1400 (0.61) 301 / 248, 2048 (0.90) 424 / 269, 4505 (0.85) 680 / 600; 2 x 5632 of
  // 2048, 1300 (0.44) 76 / 89, 1800 (0.60) 94 / 94, 3300 (0.74) 162 / 139; 2 x 13824 of 5120, 768 (0.63) 205 / 207, 1024 (0.85) 270 / 224.  The library's
  // own steps lie elsewhere: at the line this loses up to 6 % (2 x 14336 of 4096, 384 rows (0.66) 93 / 99; 2 x 13824 of 5120, 1150 (0.63) 300 / 312) and gains 20.
  const int64_t tiles = (M + kTileRows - 1) / kTileRows * ((2 * inter + kTileRows - 1) / kTileRows);
  const int64_t rounds = (tiles + kTileGroups - 1) / kTileGroups;
  return (double)M * (double)(2 * inter) >= 0.6 * (double)rounds * kTileGroups * kTileRows * kTileRows;
}

extern "C" int hx_gate_up_silu_rows(void* out, const void* x, const void* weight, int64_t M, int64_t inter, int64_t K, int64_t ldx, int64_t ldw,
                                    int dtype, hx_stream stream) {
  if (M < 0 || inter < 16 || inter % 16 || K < 2 * kTileK || K % kTileK || M > (1 << 24) || inter > (1 << 24) || K > (1 << 24)) return HX_ERR_SHAPE;
  if (M == 0) return HX_OK;
  if (!out || !x || !weight) return HX_ERR_NULL;
  if (dtype != HX_F16 && dtype != HX_BF16) return HX_ERR_DTYPE;
  if (ldx < K || ldw < K || ldx % 8 || ldw % 8 || !aligned16(out) || !aligned16(x) || !aligned16(weight)) return HX_ERR_STRIDE;
  // (32-bit byte offsets of rows and weight rows)
  if (ldx > 0x7fffffff / M || ldw > 0x7fffffff / (2 * inter)) return HX_ERR_STRIDE;
  if (gate_up_in_small_tiles(M, inter, K)) return gate_up_small_tiles(out, x, weight, M, inter, K, ldx, ldw, dtype, (hipStream_t)stream);
  const int64_t n_row = (M + kTileRows - 1) / kTileRows, n_col = (inter + kTileRows / 2 - 1) / (kTileRows / 2), tiles = n_row * n_col;
  if (tiles > 0x7fffffff) return HX_ERR_SHAPE;
  const int64_t panels = (n_row + 10) / 11;
  const unsigned grid = tiles < kTileGroups ? (unsigned)((tiles + 7) / 8 * 8) : kTileGroups;
  auto kernel = dtype == HX_F16 ? gate_up_silu_rows_kernel<F16> : gate_up_silu_rows_kernel<BF16>;
  const int rc = hip_rc(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTileLds));
  if (rc != HX_OK) return rc;
  hx::launcher(kernel, dim3(grid), dim3(256), kTileLds, (hipStream_t)stream)((u16*)out, (const u16*)x, (const u16*)weight, (int)M, (int)inter, (int)K,
                                                                            ldx, ldw, (int)((n_row + panels - 1) / panels));
  return check_launch();
}
