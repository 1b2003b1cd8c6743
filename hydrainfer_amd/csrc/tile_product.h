// tile_product.h — the inner part of products of many rows: a workgroup of four waves multiplies 256 rows by 256 weight rows
// (Y = X W^T), 64 k a slice, tile after tile without a pause.  Used by moe_mix.hip (the experts' rows) and gemm_tile.hip.
//
// A wave keeps 128 x 128 results (256 accumulators a lane, one wave a SIMD): a byte read from LDS feeds 32 multiply-adds, eight
// waves of 128 x 64 make of it 21.  Rows and weight rows come straight to LDS, 128 bytes of a row next to each other (in rows of 64
// bytes L2 serves every line twice: 8192 x 8192 x 8192 1240 us instead of 953), in a ring of five half slots of 32 KB: half a slice
// is free at any time, so that loads go out evenly, one behind every eight products, one and a half slices before they are needed.
// Every other instruction stands by itself between two products: bunched, they hold the matrix cores up (256 tiles of 8192 k,
// us a slice with data of zeros: reads and four loads in front of every eight products 1.35, two loads 1.18, dealt singly 1.05, with
// the fifth half slot 1.02; the products alone take 0.85 at 2.4 GHz).  With normal data the card's power is the bound and traffic
// costs clock: 1.34 us a slice, 1.58 PFLOP/s (32x32x16 products: 0.98 and 1.50).
// An LDS row's 16-byte chunk c sits at position c ^ (row / 2 % 8), so that the 16 lanes that one pass of a 16-byte read serves
// (rows 0-3, 12-15 of one k group and 4-11 of the next) fall into different banks.
// Products are made as W X^T: a lane holds four columns of a row, and two of them next to each other make a 16-byte store.
#pragma once
#include <type_traits>
#include "attn_common.h"

namespace hx {

constexpr int kTileRows = 256, kTileK = 64;
constexpr uint32_t kTileHalf = kTileRows * kTileK * 2;      // bytes of a half slot: a slice of the rows or of the weight rows
constexpr size_t kTileLds = 5 * kTileHalf;
constexpr int kTileGroups = 256;                            // workgroups that run at a time: one a CU

template <int N>
__device__ __forceinline__ void tile_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// Where a lane's 16 bytes of load j of a wave come from: row of the tile, element within the slice (they land lane after lane).
__device__ __forceinline__ int tile_load_row(int wave, int j, int lane) { return 64 * wave + 8 * j + (lane >> 3); }
__device__ __forceinline__ int tile_load_k(int j, int lane) { return 8 * ((lane & 7) ^ (((j & 1) << 2) + (lane >> 4))); }

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// 1 KB from base + offset (bytes, each lane's own) or from at to LDS address lds + 1024 J.  (m0, the address of the transfer, is a
// reserved register: nothing else in these kernels uses it.)
template <int J>
__device__ __forceinline__ void tile_load(const u16* base, uint32_t offset, uint32_t lds) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(offset), "s"(base), "s"(lds), "n"(J * 1024) : "m0", "scc");
}
template <int J>
__device__ __forceinline__ void tile_load(const u16* at, uint32_t lds) {
  asm volatile("s_add_u32 m0, %1, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(at), "s"(lds), "n"(J * 1024) : "m0", "scc");
}
#pragma clang diagnostic pop

// T: F16 or BF16.  Loader: a<J>(lds), b<J>(lds) request load J (0 .. 7) of the stream's next slice of rows or weight rows (all eight
// are requested in order; behind the eighth the loader goes on to the next slice, of the next tile behind a tile's last).
template <typename T, typename Loader>
struct TileProduct {
  struct Frags {
    u16x8 w[8], x[8];
  };
  f32x4 acc[8][8];                // [16 rows][16 columns]: lane l holds columns 4 (l / 16) .. + 3 of row l % 16
  Frags f0, f1;
  Loader& loader;
  char* smem;
  uint32_t lds, a0, b0, a1, b1, a2;      // half slots: this slice, the next, the rows of the one behind it
  int x_at, w_at;                 // where this lane's first operand starts in a half slot

  __device__ __forceinline__ TileProduct(char* smem_, Loader& loader_) : loader(loader_), smem(smem_) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = threadIdx.x & 15;
    lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem + wave * 8192;
    x_at = ((wave >> 1) * 128 + l16) * 128;
    w_at = ((wave & 1) * 128 + l16) * 128;
    a0 = 0, b0 = kTileHalf, a1 = 2 * kTileHalf, b1 = 3 * kTileHalf, a2 = 4 * kTileHalf;
    clear();
  }
  // (the accumulators change places with other registers here only: left to the compiler, all 256 of them are copied, and spilled,
  // wherever a branch stands between the products and the stores)
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) asm volatile("v_accvgpr_write_b32 %0, 0" : "=a"(acc[i][j][q]));
  }
  __device__ __forceinline__ f32x4 take(int i, int j) {
    asm volatile("" : "+a"(acc[i][j]));
    return acc[i][j];
  }
  template <int N>
  __device__ __forceinline__ void read(Frags& f, uint32_t a, uint32_t b, int half) {
    const int chunk = ((4 * half + ((threadIdx.x >> 4) & 3)) ^ ((threadIdx.x >> 1) & 7)) * 16;
    if constexpr (N < 8) f.w[N] = *reinterpret_cast<const u16x8*>(smem + b + w_at + chunk + N * 2048);
    else f.x[N - 8] = *reinterpret_cast<const u16x8*>(smem + a + x_at + chunk + (N - 8) * 2048);
  }
  __device__ __forceinline__ void multiply(const Frags& f, int i, int j) { acc[i][j] = Mfma<T>::mma(f.w[j], f.x[i], acc[i][j]); }
  template <int... I>
  __device__ __forceinline__ void read_all(Frags& f, uint32_t a, uint32_t b, int half, std::integer_sequence<int, I...>) { (read<I>(f, a, b, half), ...); }
  template <int... J>
  __device__ __forceinline__ void load_a(uint32_t slot, std::integer_sequence<int, J...>) { (loader.template a<J>(lds + slot), ...); }
  template <int... J>
  __device__ __forceinline__ void load_b(uint32_t slot, std::integer_sequence<int, J...>) { (loader.template b<J>(lds + slot), ...); }

  // Half a slice: the products of `now`, between them the reads of the next half and eight loads (of rows, or of weight rows)
  template <bool ROWS, int U>
  __device__ __forceinline__ void unit(const Frags& now, Frags& next, uint32_t a, uint32_t b, int half, uint32_t to) {
    if constexpr (U % 3 == 0 && U / 3 < 16) read<U / 3>(next, a, b, half);
    if constexpr (U % 8 == 1) {
      if constexpr (ROWS) loader.template a<U / 8>(lds + to);
      else loader.template b<U / 8>(lds + to);
    }
    multiply(now, U / 8, U % 8);
    __builtin_amdgcn_sched_barrier(0);
  }
  template <bool ROWS, int... U>
  __device__ __forceinline__ void half_slice(const Frags& now, Frags& next, uint32_t a, uint32_t b, int half, uint32_t to, std::integer_sequence<int, U...>) {
    (unit<ROWS, U>(now, next, a, b, half, to), ...);
  }

  // The stream's first two slices on their way and the first half of the first in registers
  __device__ __forceinline__ void start() {
    typedef std::make_integer_sequence<int, 8> Eight;
    load_a(a0, Eight());
    load_b(b0, Eight());
    load_a(a1, Eight());
    load_b(b1, Eight());
    tile_wait<16>();
    barrier();
    read_all(f0, a0, b0, 0, std::make_integer_sequence<int, 16>());
  }
  // One slice of the stream; the slice two behind it is requested, the first half of the next read.
  __device__ __forceinline__ void slice() {
    typedef std::make_integer_sequence<int, 64> Units;
    half_slice<true>(f0, f1, a0, b0, 1, a2, Units());
    // the next slice is there when only the rows just requested are on their way; past the barrier every wave's part of it is, and
    // every wave has read all of this one: its half slots can be filled again
    tile_wait<8>();
    barrier();
    __builtin_amdgcn_sched_barrier(0);
    half_slice<false>(f1, f0, a1, b1, 0, a0, Units());
    const uint32_t free_a = a0, free_b = b0;
    a0 = a1, b0 = b1, a1 = a2, b1 = free_a, a2 = free_b;
  }
  // (orders LDS traffic only: loads stay in flight)
  __device__ __forceinline__ void barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  }
};

// Two 16-column results of a row (columns 4 g .. + 3 of each in lane group g) as 8 columns in a lane: returns them, and the first
// one's column relative to the pair's
__device__ __forceinline__ u32x4 tile_pair(u32x2 first, u32x2 second) {
  const auto lo = __builtin_amdgcn_permlane16_swap(first[0], second[0], false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(first[1], second[1], false, false);
  return u32x4{lo[0], hi[0], lo[1], hi[1]};
}
__device__ __forceinline__ int tile_pair_column(int lane) { return 16 * ((lane >> 4) & 1) + 8 * (lane >> 5); }
template <typename T>
__device__ __forceinline__ u32x2 tile_round(f32x4 v) {
  return u32x2{(uint32_t)T::from_float(v[0]) | (uint32_t)T::from_float(v[1]) << 16, (uint32_t)T::from_float(v[2]) | (uint32_t)T::from_float(v[3]) << 16};
}

}  // namespace hx
