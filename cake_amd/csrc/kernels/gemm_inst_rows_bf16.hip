// Instantiates the products of few rows (gemm_rows.h) for bf16.
#include "gemm_rows.h"

template struct cake::Rows<cake::kBF16>;
