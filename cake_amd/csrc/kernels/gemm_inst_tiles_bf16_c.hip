// Instantiates the four-wave tiles of CAKE_GEMM_4W_TILES (gemm_4w.h) for bf16, epilogues Quick, Gelu, Relu2;
// split from gemm.hip so the heavy instantiations compile in parallel.
#include "gemm_kernel.h"

namespace cake {
template int launch_tiles<kBF16, kEpiQuick, false>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_tiles<kBF16, kEpiQuick, true>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_tiles<kBF16, kEpiGelu, false>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_tiles<kBF16, kEpiGelu, true>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_tiles<kBF16, kEpiRelu2, false>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_tiles<kBF16, kEpiRelu2, true>(int, dim3, hipStream_t, const GemmArgs&);
}  // namespace cake
