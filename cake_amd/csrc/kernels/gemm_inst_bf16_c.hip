// Instantiates the GEMM launchers (gemm_kernel.h) for bf16, epilogues Quick, Gelu, Relu2;
// split from gemm.hip so the heavy instantiations compile in parallel.
#include "gemm_kernel.h"

namespace cake {
template int launch_gemm<kBF16, kEpiQuick>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_gemm<kBF16, kEpiGelu>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_gemm<kBF16, kEpiRelu2>(int, dim3, hipStream_t, const GemmArgs&);
}  // namespace cake
