// Instantiates the four-wave tiles of CAKE_GEMM_4W_TILES (gemm_4w.h) for f16, epilogues Swiglu, Store32, Silu;
// split from gemm.hip so the heavy instantiations compile in parallel.
#include "gemm_kernel.h"

namespace cake {
template int launch_tiles<kF16, kEpiSwiglu, false>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_tiles<kF16, kEpiSwiglu, true>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_tiles<kF16, kEpiStore32, false>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_tiles<kF16, kEpiStore32, true>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_tiles<kF16, kEpiSilu, false>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_tiles<kF16, kEpiSilu, true>(int, dim3, hipStream_t, const GemmArgs&);
}  // namespace cake
