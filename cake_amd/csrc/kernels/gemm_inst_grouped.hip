// Grouped products: rows sorted by weight group (routed experts), every row tile reading its own
// group's weight.  Tiles of gemm_ws.h (64 rows and fewer: gemm_kernel.h) with the tile list as their row map.
#include <algorithm>

#include "gemm_kernel.h"

namespace cake {

constexpr long long kWide = 1 << 22;  // elements: 256 rows of this stride are 2 GB

// Tiles by rows; cfg 4: 64 x 64; cfg 6: as the tile list says
constexpr int kByList = 6;
constexpr int grouped_rows(int cfg) {
  return cfg == 4 ? 64 : cfg == 0 ? 128 : cfg == 1 ? 160 : cfg == 2 ? 192 : cfg == 3 ? 224
         : cfg == 5 || cfg == kByList ? 256 : 0;
}

// One kernel for all heights, so that the one that fits the groups can be chosen on the device, where their sizes are
// known (mixer_experts.hip).  Of few tiles narrower ones, which more CUs have a share of (8 experts 4096 -> 2048 at 100 rows
// 60 us on 160 x 256, 47 on 160 x 128).  Up and down of 64 experts 4096 x 3648 at 100 / 192 even / 192 independent
// rows 400 + 383 / 444 + 436 / 476 + 463 us on gemm_4w.h's tiles, 334 + 344 / 370 + 371 / 400 + 386 here (weights at 5.7 /
// 5.1 / 4.9 TB/s); of 14 expert sizes at 70 .. 600 rows, even and skewed, 1.14 times as fast on the average.
template <int DT, int EPI>
__global__ __launch_bounds__((WsTile<160, 256>::THREADS)) void gemm_groups_kernel(GemmArgs g) {
  constexpr int MOST = std::max({WsTile<160, 256>::LDS, WsTile<192, 256>::LDS, WsTile<224, 256>::LDS, WsTile<256, 256>::LDS,
                                 WsTile<160, 128>::LDS, WsTile<256, 128>::LDS});
  __shared__ __attribute__((aligned(16))) uint8_t smem[MOST];
  const int rows = uni(g.pieces > 0 ? g.pieces : g.groups[g.tiles_m].y);
  const bool few = uni(g.groups[g.tiles_m].x) * ((g.N + 255) / 256) <= (rows <= 160 ? 128 : 64);
  g.pieces = 0;
  if (few && rows <= 160) ws_tiles<DT, EPI, 160, 128, true>(g, smem);
  else if (few) ws_tiles<DT, EPI, 256, 128, true>(g, smem);
  else if (rows <= 160) ws_tiles<DT, EPI, 160, 256, true>(g, smem);
  else if (rows <= 192) ws_tiles<DT, EPI, 192, 256, true>(g, smem);
  else if (rows <= 224) ws_tiles<DT, EPI, 224, 256, true>(g, smem);
  else ws_tiles<DT, EPI, 256, 256, true>(g, smem);
}

// The same on four waves (gemm_4w.h), for rows of kGroupedShort k and fewer: 16 steps do not make up for the longer start of the
// other (64 experts 1024 x 1024 at 100 rows 32 us, 34; 32 of 1024 -> 2816 47, 51).  All heights fill a CU's LDS alone: a
// branch over whole bodies costs none of them a workgroup.  A tile runs at the least height that holds its rows.
template <int DT, int EPI>
__global__ __launch_bounds__(256) void gemm_heights_kernel(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) uint8_t smem[FourWave<160, 256, 2>::NBUF * FourWave<160, 256, 2>::BUF];
  const int n = g.groups[g.tiles_m].x;
  if ((int)blockIdx.x >= n * g.tiles_n) return;
  const int most = g.pieces > 0 ? g.pieces : g.groups[g.tiles_m].y;
  const int tm = grouped_place(n, g.tiles_n, blockIdx.x).x;
  const int has = min(__builtin_amdgcn_readfirstlane(g.groups[tm].z), __builtin_amdgcn_readfirstlane(most));
  const int rows = has <= 128 ? 128 : has <= 160 ? 160 : has <= 192 ? 192 : 256;
#define X(BM, SCHED)                                                                         \
  if (rows == BM) {                                                                          \
    static_assert(FourWave<BM, 256, SCHED>::NBUF * FourWave<BM, 256, SCHED>::BUF <= (int)sizeof(smem), "LDS"); \
    gemm_4w_tile<DT, EPI, BM, 256, SCHED, true, false>(g, smem);                             \
    return;                                                                                  \
  }
  X(128, 2) X(160, 2) X(192, 1) X(256, 1)
#undef X
}

// Rows too far apart for 32-bit offsets take the 64-row tile, in passes.
template <int DT, int EPI>
static int launch_grouped(int cfg, int tiles, hipStream_t st, GemmArgs& g) {
  const int bm = grouped_rows(cfg);
  const bool wide = g.lda >= kWide || g.ldb >= kWide;
  if (bm == 64 || wide) {
    g.tiles_n = (g.N + 63) / 64;
    const dim3 grid(tiles * g.tiles_n, wide ? (bm + 63) / 64 : 1);
    hipLaunchKernelGGL((gemm_kernel<DT, 64, 64, 2, 2, 2, EPI, 6, true>), grid, dim3(256), 0, st, g);
    return (int)hipGetLastError();
  }
  g.pieces = cfg == kByList ? 0 : bm;   // rows of a tile
  if (g.K <= kGroupedShort) {
    g.tiles_n = (g.N + 255) / 256;
    hipLaunchKernelGGL((gemm_heights_kernel<DT, EPI>), dim3(tiles * g.tiles_n), dim3(256), 0, st, g);
    return (int)hipGetLastError();
  }
  const int grid = (int)std::min(256LL, (long long)tiles * ((g.N + 127) / 128));
  hipLaunchKernelGGL((gemm_groups_kernel<DT, EPI>), dim3(grid), dim3(WsTile<160, 256>::THREADS), 0, st, g);
  return (int)hipGetLastError();
}

}  // namespace cake

using namespace cake;

// c[row0 + r] = act(a[row0 + r] W[group]^T) over the tiles [group, row0, rows, 0] (0 < rows <= the
// configuration's BM), at most max_tiles of them; entry max_tiles of the list is [count, BM, 0, 0] (BM, 128 to
// 256, read in configuration 6 only).
// epi 0: no activation, 7 .. 10 as cake_gemm_scaled.  K % 8 == 0.
CAKE_API int cake_gemm_grouped(int dt, int epi, int cfg, const void* a, long long lda, const void* b,
                               long long ldb, long long b_group, void* c, long long ldc,
                               const void* tiles, int max_tiles, const void* zeros, int N, int K,
                               hipStream_t st) {
  if (max_tiles <= 0 || N <= 0 || K <= 0 || K % 8 || lda % 8 || ldb % 8 || b_group % 8 ||
      !(epi == 0 || (epi >= 7 && epi <= 10)) || grouped_rows(cfg) == 0)
    return (int)hipErrorInvalidValue;
  GemmArgs g{};
  g.a = (const uint16_t*)a; g.b = (const uint16_t*)b; g.c = (uint16_t*)c;
  g.zeros = (const uint16_t*)zeros;
  g.lda = lda; g.ldb = ldb; g.ldc = ldc;
  g.N = N; g.K = K; g.Nv = N; g.half = N;
  g.tiles_m = max_tiles;
  g.kps = (K + kGBK - 1) / kGBK * kGBK;
  g.groups = (const int4*)tiles;
  g.b_group = b_group;
  const auto run = [&](auto dtc) {
    constexpr int DT = decltype(dtc)::value;
    switch (epi) {
      case kEpiStore: return launch_grouped<DT, kEpiStore>(cfg, max_tiles, st, g);
      case kEpiSilu: return launch_grouped<DT, kEpiSilu>(cfg, max_tiles, st, g);
      case kEpiQuick: return launch_grouped<DT, kEpiQuick>(cfg, max_tiles, st, g);
      case kEpiGelu: return launch_grouped<DT, kEpiGelu>(cfg, max_tiles, st, g);
      case kEpiRelu2: return launch_grouped<DT, kEpiRelu2>(cfg, max_tiles, st, g);
    }
    return (int)hipErrorInvalidValue;
  };
  return dt == kBF16 ? run(std::integral_constant<int, kBF16>{})
         : dt == kF16 ? run(std::integral_constant<int, kF16>{}) : (int)hipErrorInvalidValue;
}
