// Instantiates the four-wave tiles in pieces (gemm_4w.h) for bf16, epilogues Store, Resid32, Add16, Swiglu, Geglu;
// split from gemm.hip so the heavy instantiations compile in parallel.
#include "gemm_kernel.h"

namespace cake {
template int launch_pieces<kBF16, kEpiStore>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_pieces<kBF16, kEpiResid32>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_pieces<kBF16, kEpiAdd16>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_pieces<kBF16, kEpiSwiglu>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_pieces<kBF16, kEpiGeglu>(int, dim3, hipStream_t, const GemmArgs&);
}  // namespace cake
