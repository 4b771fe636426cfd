// Grouped products: rows sorted by weight group (routed experts), every row tile reading its own
// group's weight.  The plain GEMM's tiles (gemm_kernel.h, gemm_4w.h) with the tile list as their row
// map.
#include "gemm_kernel.h"

namespace cake {

constexpr long long kWide = 1 << 22;  // elements: 256 rows of this stride are 2 GB

// Tiles by rows, of 256 columns on four waves (gemm_4w.h); cfg 4: 64 x 64; cfg 6: as the tile list says
constexpr int kByList = 6;
constexpr int grouped_rows(int cfg) {
  return cfg == 4 ? 64 : cfg == 0 ? 128 : cfg == 1 ? 160 : cfg == 2 ? 192 : cfg == 5 || cfg == kByList ? 256 : 0;
}

// One kernel for the four heights, so that the one that fits the groups can be chosen on the device, where
// their sizes are known (mixer_experts.hip).  All of them fill a CU's LDS alone: a branch over whole
// bodies costs none of them a workgroup (two products of 64 experts 4096 x 3648, 192 rows each: 932 us in
// a kernel of its own, 938 so; over all heights and seven sizes 0.8 % more).  A tile runs at the least height
// that holds its rows, the list's is what the longest of them needs: of 44 pairs of products, even and skewed groups of
// 70 .. 600 rows, up to 12 % faster, 1.2 % on the average (64 of 4096 x 3648 at 170 rows 488 + 463 us, 451 + 429;
// eight of 4096 x 4096 at 300 rows 93 + 91, 81 + 81), none slower by more than they vary.
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

// Rows too far apart for the four waves' 32-bit offsets take the 64-row tile, in passes.
template <int DT, int EPI>
static int launch_grouped(int cfg, int tiles, hipStream_t st, GemmArgs& g) {
  const int bm = grouped_rows(cfg);
  const bool wide = g.lda >= kWide || g.ldb >= kWide;
  const int bn = bm == 64 || wide ? 64 : 256;
  g.tiles_n = (g.N + bn - 1) / bn;
  const dim3 grid(tiles * g.tiles_n, wide ? (bm + 63) / 64 : 1);
  if (bn == 64) {
    hipLaunchKernelGGL((gemm_kernel<DT, 64, 64, 2, 2, 2, EPI, 6, true>), grid, dim3(256), 0, st, g);
    return (int)hipGetLastError();
  }
  g.pieces = cfg == kByList ? 0 : bm;   // rows of a tile
  hipLaunchKernelGGL((gemm_heights_kernel<DT, EPI>), grid, dim3(256), 0, st, g);
  return (int)hipGetLastError();
}

}  // namespace cake

using namespace cake;

// c[row0 + r] = act(a[row0 + r] W[group]^T) over the tiles [group, row0, rows, 0] (0 < rows <= the
// configuration's BM), at most max_tiles of them; entry max_tiles of the list is [count, BM, 0, 0] (BM, 128,
// 160, 192 or 256, read in configuration 6 only).
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
