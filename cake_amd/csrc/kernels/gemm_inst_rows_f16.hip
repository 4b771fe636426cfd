// Instantiates the products of few rows (gemm_rows.h) for f16.
#include "gemm_rows.h"

namespace cake {
#define X(E) template int launch_rows<kF16, E>(int, int, dim3, hipStream_t, const GemmArgs&);
X(kEpiStore) X(kEpiResid32) X(kEpiAdd16) X(kEpiSwiglu) X(kEpiGeglu) X(kEpiStore32) X(kEpiSilu)
#undef X
template int launch_rows_grouped<kF16, kEpiStore>(int, dim3, hipStream_t, const GemmArgs&);
template int launch_rows_grouped<kF16, kEpiSilu>(int, dim3, hipStream_t, const GemmArgs&);
}  // namespace cake
