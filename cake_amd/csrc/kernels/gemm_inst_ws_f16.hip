// Instantiates the tiles of gemm_ws.h for f16: f32 results, whole tiles and pieces.
#include "gemm_kernel.h"

namespace cake {
template int launch_ws<kF16, kEpiResid32>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_ws<kF16, kEpiStore32>(int, dim3, hipStream_t, const GemmArgs&);
}  // namespace cake
