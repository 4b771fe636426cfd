// Instantiates the four-wave tiles in pieces (gemm_4w.h) for bf16, epilogues Store32, Silu, Quick, Gelu, Relu2;
// split from gemm.hip so the heavy instantiations compile in parallel.
#include "gemm_kernel.h"

namespace cake {
template int launch_pieces<kBF16, kEpiStore32>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_pieces<kBF16, kEpiSilu>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_pieces<kBF16, kEpiQuick>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_pieces<kBF16, kEpiGelu>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_pieces<kBF16, kEpiRelu2>(int, dim3, hipStream_t, const GemmArgs&);
}  // namespace cake
