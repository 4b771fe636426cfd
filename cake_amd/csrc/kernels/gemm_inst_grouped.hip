// Grouped products: rows sorted by weight group (routed experts), every row tile reading its own
// group's weight.  The plain GEMM's tiles (gemm_kernel.h) with the tile list as their row map.
#include "gemm_kernel.h"

namespace cake {

template <int DT, int EPI>
static int launch_grouped(int cfg, dim3 grid, hipStream_t st, const GemmArgs& g) {
#define X(id, BM, BN, WM, WN, NS, PR)                                                      \
  if (cfg == id) {                                                                         \
    hipLaunchKernelGGL((gemm_kernel<DT, BM, BN, WM, WN, NS, EPI, PR, true>), grid,         \
                       dim3(64 * WM * WN), 0, st, g);                                      \
    return (int)hipGetLastError();                                                         \
  }
  X(0, 128, 128, 2, 2, 2, 6)
  X(4, 64, 64, 2, 2, 2, 6)
  X(5, 256, 256, 2, 4, 2, 6)
#undef X
  return (int)hipErrorInvalidValue;
}

}  // namespace cake

using namespace cake;

// c[row0 + r] = act(a[row0 + r] W[group]^T) over the tiles [group, row0, rows, 0] (0 < rows <= the
// configuration's BM), at most max_tiles of them; entry max_tiles of the list is [count, 0, 0, 0].
// epi 0: no activation, 7 .. 10 as cake_gemm_scaled.  K % 8 == 0.
CAKE_API int cake_gemm_grouped(int dt, int epi, int cfg, const void* a, long long lda, const void* b,
                               long long ldb, long long b_group, void* c, long long ldc,
                               const void* tiles, int max_tiles, const void* zeros, int N, int K,
                               hipStream_t st) {
  if (max_tiles <= 0 || N <= 0 || K <= 0 || K % 8 || lda % 8 || ldb % 8 || b_group % 8 ||
      !(epi == 0 || (epi >= 7 && epi <= 10)))
    return (int)hipErrorInvalidValue;
  const int bn = cfg == 4 ? 64 : cfg == 5 ? 256 : 128;
  GemmArgs g{};
  g.a = (const uint16_t*)a; g.b = (const uint16_t*)b; g.c = (uint16_t*)c;
  g.zeros = (const uint16_t*)zeros;
  g.lda = lda; g.ldb = ldb; g.ldc = ldc;
  g.N = N; g.K = K; g.Nv = N; g.half = N;
  g.tiles_m = max_tiles;
  g.tiles_n = (N + bn - 1) / bn;
  g.kps = (K + kGBK - 1) / kGBK * kGBK;
  g.groups = (const int4*)tiles;
  g.b_group = b_group;
  const dim3 grid(g.tiles_m * g.tiles_n, 1);
  const auto run = [&](auto dtc) {
    constexpr int DT = decltype(dtc)::value;
    switch (epi) {
      case kEpiStore: return launch_grouped<DT, kEpiStore>(cfg, grid, st, g);
      case kEpiSilu: return launch_grouped<DT, kEpiSilu>(cfg, grid, st, g);
      case kEpiQuick: return launch_grouped<DT, kEpiQuick>(cfg, grid, st, g);
      case kEpiGelu: return launch_grouped<DT, kEpiGelu>(cfg, grid, st, g);
      case kEpiRelu2: return launch_grouped<DT, kEpiRelu2>(cfg, grid, st, g);
    }
    return (int)hipErrorInvalidValue;
  };
  return dt == kBF16 ? run(std::integral_constant<int, kBF16>{})
         : dt == kF16 ? run(std::integral_constant<int, kF16>{}) : (int)hipErrorInvalidValue;
}
