// prompt_rows.hip — the rows of a batch of prompts that are sampled, taken out in front of the last layer's queries (extends
// hydrainfer/model/model_forward.py, where they are taken out in front of its feed-forward): behind that layer's keys and values no other row is used.
#include "hx_common.h"
#include "../../include/hydra_hip.h"

namespace hx {
namespace {

struct PromptRows {
  const void* rows;               // [n] int32 or int64; negative ones count from the end
  int32_t wide, n, n_tokens, n_seq;
  const int32_t *q_cu, *kv_cu, *cu_blocks, *positions;
  const u16 *x, *h;
  u16 *x_out, *h_out;
  int32_t row_bytes;
  int32_t *position_out, *q_cu_out, *kv_cu_out, *cu_blocks_out;
};

__device__ __forceinline__ int prompt_row(const PromptRows& p, int i) {
  const int64_t r = p.wide ? ((const int64_t*)p.rows)[i] : ((const int32_t*)p.rows)[i];
  const int64_t at = r < 0 ? r + p.n_tokens : r;
  return (int)(at < 0 ? 0 : at >= p.n_tokens ? p.n_tokens - 1 : at);
}

// Workgroup i < n: row i of both; the last one: each row as a sequence of one query, with the keys that it sees.
__global__ __launch_bounds__(256) void prompt_rows_kernel(PromptRows p) {
  const int tid = threadIdx.x;
  if ((int)blockIdx.x < p.n) {
    const int64_t from = (int64_t)prompt_row(p, blockIdx.x) * p.row_bytes, to = (int64_t)blockIdx.x * p.row_bytes;
    for (int c = 16 * tid; c < p.row_bytes; c += 16 * 256) {
      *reinterpret_cast<u32x4*>((char*)p.x_out + to + c) = *reinterpret_cast<const u32x4*>((const char*)p.x + from + c);
      *reinterpret_cast<u32x4*>((char*)p.h_out + to + c) = *reinterpret_cast<const u32x4*>((const char*)p.h + from + c);
    }
    return;
  }
  __shared__ int32_t sums[4];
  int32_t run = 0;                // keys of the rows in front
  for (int i0 = 0; i0 < p.n; i0 += 256) {
    const int i = i0 + tid;
    int32_t keys = 0;
    if (i < p.n) {
      const int r = prompt_row(p, i);
      int lo = 0, hi = p.n_seq - 1;                        // the last sequence that starts at or before row r
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (p.q_cu[mid] <= r) lo = mid;
        else hi = mid - 1;
      }
      keys = p.kv_cu[lo + 1] - p.kv_cu[lo] - (p.q_cu[lo + 1] - 1 - r);
      p.position_out[i] = p.positions[r];
      p.q_cu_out[i] = i;
      p.cu_blocks_out[i] = p.cu_blocks[lo];
    }
    int32_t up_to = keys;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t v = __shfl_up(up_to, d, 64);
      if ((tid & 63) >= d) up_to += v;
    }
    if ((tid & 63) == 63) sums[tid >> 6] = up_to;
    __syncthreads();
    for (int w = 0; w < 4; ++w) {
      if (w < tid >> 6) up_to += sums[w];
    }
    if (i < p.n) p.kv_cu_out[i] = run + up_to - keys;
    run += sums[0] + sums[1] + sums[2] + sums[3];
    __syncthreads();
  }
  if (tid == 0) {
    p.q_cu_out[p.n] = p.n;
    p.kv_cu_out[p.n] = run;
    p.cu_blocks_out[p.n] = p.cu_blocks[p.n_seq];
  }
}

}  // namespace
}  // namespace hx

using namespace hx;

extern "C" int hx_prompt_rows(const void* rows, int32_t rows_are_int64, int64_t n, int64_t n_tokens, int64_t n_seq, const int32_t* q_cu, const int32_t* kv_cu, const int32_t* cu_blocks,
                              const int32_t* positions, const void* x, const void* h, void* x_out, void* h_out, int64_t row_bytes, int32_t* tables, hx_stream stream) {
  if (n < 0 || n > 65535 || n_tokens < 1 || n_tokens > INT32_MAX || n_seq < 1 || n_seq > 65535 || row_bytes < 16 || row_bytes % 16 || row_bytes > (1 << 20)) return HX_ERR_SHAPE;
  if (n == 0) return HX_OK;
  if (!rows || !q_cu || !kv_cu || !cu_blocks || !positions || !x || !h || !x_out || !h_out || !tables) return HX_ERR_NULL;
  if (!aligned16(x) || !aligned16(h) || !aligned16(x_out) || !aligned16(h_out)) return HX_ERR_STRIDE;
  PromptRows p;
  p.rows = rows; p.wide = rows_are_int64 != 0; p.n = (int32_t)n; p.n_tokens = (int32_t)n_tokens; p.n_seq = (int32_t)n_seq;
  p.q_cu = q_cu; p.kv_cu = kv_cu; p.cu_blocks = cu_blocks; p.positions = positions;
  p.x = (const u16*)x; p.h = (const u16*)h; p.x_out = (u16*)x_out; p.h_out = (u16*)h_out; p.row_bytes = (int32_t)row_bytes;
  p.q_cu_out = tables; p.kv_cu_out = tables + (n + 1); p.cu_blocks_out = tables + 2 * (n + 1); p.position_out = tables + 3 * (n + 1);
  hx::launcher(prompt_rows_kernel, dim3((unsigned)(n + 1)), dim3(256), 0, (hipStream_t)stream)(p);
  return check_launch();
}
