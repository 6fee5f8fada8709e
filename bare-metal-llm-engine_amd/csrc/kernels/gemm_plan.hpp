// gemm_plan.hpp -- tile numbering and the stream-K plan shared by the GEMM kernels.
#pragma once

#include "../engine_internal.hpp"

namespace eng {
namespace {

constexpr int kGroupM = 8;  // tile-rows per raster group
constexpr int kXcds = 8;

// Workgroup id -> (tile_m, tile_n). Workgroups are handed to XCDs round-robin,
// so id w runs on XCD w % 8; renumber so XCD x gets a contiguous logical range,
// then raster that range in groups of kGroupM tile-rows.
__device__ __forceinline__ void tile_of(int wg, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int ntiles = tiles_m * tiles_n;
  const int q = ntiles / kXcds;
  const int r = ntiles % kXcds;
  const int xcd = wg % kXcds;
  const int local = wg / kXcds;
  const int logical = xcd * q + (xcd < r ? xcd : r) + local;
  const int group_size = kGroupM * tiles_n;
  const int group = logical / group_size;
  const int first_m = group * kGroupM;
  const int gm = (tiles_m - first_m) < kGroupM ? (tiles_m - first_m) : kGroupM;
  const int in_group = logical - group * group_size;
  tm = first_m + in_group % gm;
  tn = in_group / gm;
}

// Stream-K plan: of T tiles in tile_of order the first `dp` are computed whole
// by workgroups 0 .. dp - 1, and the remaining T - dp tiles' K iterations are
// split evenly over workgroups dp .. dp + nsk - 1: workgroup dp + s takes
// iterations [s I / nsk, (s + 1) I / nsk) of the tail's I = (T - dp) nk, tile by
// tile. A tail tile one workgroup covers whole is stored to C; a split tile
// leaves one record per workgroup (slot 0 its first tile, slot 1 its last),
// which gemm_sk_fixup_kernel adds in workgroup order.
struct SkPlan {
  int dp = 0;        // data-parallel tiles
  int nsk = 0;       // stream-K workgroups
  int nk = 0;        // K tiles per output tile
  long long I = 0;   // tail iterations (tail tiles x nk)
};

__host__ __device__ inline long long sk_begin(long long s, const SkPlan& p) {
  return s * p.I / p.nsk;
}

// sk_begin for the fix-up kernel, which needs several per thread: a 64-bit
// division takes over 100 instructions there, and s I fits 32 bits unless the
// tail holds millions of K tiles.
__device__ inline long long sk_begin_fast(long long s, const SkPlan& p) {
  const long long n = s * p.I;
  if ((n >> 32) == 0) return static_cast<unsigned>(n) / static_cast<unsigned>(p.nsk);
  return n / p.nsk;
}

// Stream-K workgroup whose range holds tail iteration it.
__device__ inline long long sk_worker(long long it, const SkPlan& p) {
  const long long n = it * p.nsk + p.nsk - 1;
  long long s =
      ((n | p.I) >> 32) == 0 ? static_cast<unsigned>(n) / static_cast<unsigned>(p.I) : n / p.I;
  if (s >= p.nsk) s = p.nsk - 1;
  while (s + 1 < p.nsk && sk_begin_fast(s + 1, p) <= it) ++s;
  while (s > 0 && sk_begin_fast(s, p) > it) --s;
  return s;
}

// Split tail tiles: C = the tile's records added in workgroup order. One
// block per (tail tile, 1024 elements); tiles one workgroup covered whole are
// skipped (already stored). Bound by the records' read: 512 x 4096 x 4096 in 256
// x 128 tiles split four ways (33 MB) 11.2 -> 9 us with 32-bit plan arithmetic
// and the four loads in flight together; with many records to a tile by the number
// of loads in flight and by the arithmetic between them (70 x 56 x 8190, 32 records:
// the call 14.8 us in clamped groups of four, 17.3 of eight, 12.8 so).
template <int BM, int BN, bool EDGE = false>
__global__ __launch_bounds__(256) void gemm_sk_fixup_kernel(const float* __restrict__ rec,
                                                            float* __restrict__ C, int M, int N,
                                                            int tiles_m, int tiles_n,
                                                            SkPlan plan) {
  typedef float floatx4 __attribute__((ext_vector_type(4)));
  const long long t = blockIdx.x;
  const long long sf = sk_worker(t * plan.nk, plan);
  const long long sl = sk_worker(t * plan.nk + plan.nk - 1, plan);
  if (sf == sl) return;
  // workgroups after sf start inside the tile (slot 0); sf only when it
  // starts exactly at the tile
  const int slot_f = sk_begin_fast(sf, plan) == t * plan.nk ? 0 : 1;
  const int e = 4 * (static_cast<int>(blockIdx.y) * 256 + static_cast<int>(threadIdx.x));
  // The first record, then the others, a constant stride apart: eight loads in
  // flight together while there are so many, then up to four (past the last one it
  // again). The adds keep workgroup order.
  constexpr long long kRec = BM * BN;
  floatx4 v = *reinterpret_cast<const floatx4*>(rec + (2 * sf + slot_f) * kRec + e);
  const float* p = rec + 2 * (sf + 1) * kRec + e;
  int left = static_cast<int>(sl - sf);
  for (; left >= 8; left -= 8, p += 16 * kRec) {
    floatx4 r[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = *reinterpret_cast<const floatx4*>(p + 2 * i * kRec);
#pragma unroll
    for (int i = 0; i < 8; ++i) v += r[i];
  }
  for (; left > 0; left -= 4, p += 8 * kRec) {
    floatx4 r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      r[i] = *reinterpret_cast<const floatx4*>(p + 2 * (i < left ? i : left - 1) * kRec);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < left) v += r[i];
  }
  int tm, tn;
  tile_of(plan.dp + static_cast<int>(t), tiles_m, tiles_n, tm, tn);
  const int row = tm * BM + e / BN;
  const int col = tn * BN + e % BN;
  float* dst = C + static_cast<long long>(row) * N + col;
  if constexpr (!EDGE) {
    *reinterpret_cast<floatx4*>(dst) = v;
  } else if (row < M) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (col + q < N) dst[q] = v[q];
  }
}

template <int BM, int BN>
void launch_sk_fixup(const float* rec, float* C, int M, int N, int tiles_m, int tiles_n, int tail,
                     const SkPlan& plan, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(tail), BM * BN / 1024);
  if (M % BM == 0 && N % BN == 0 && N % 4 == 0)
    gemm_sk_fixup_kernel<BM, BN, false><<<grid, 256, 0, stream>>>(rec, C, M, N, tiles_m, tiles_n, plan);
  else
    gemm_sk_fixup_kernel<BM, BN, true><<<grid, 256, 0, stream>>>(rec, C, M, N, tiles_m, tiles_n, plan);
  ENG_LAUNCH_CHECK();
}

}  // namespace
}  // namespace eng
