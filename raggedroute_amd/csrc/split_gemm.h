// Grouped FP32 GEMM on the BF16 matrix cores (split_gemm.hip).
#pragma once

#include <hip/hip_runtime_api.h>

#include "tiles.h"

namespace rr::kern {

// Whether the split kernel can compute this problem (chain: dense_rows = rows of X).
bool split_gemm_fits(const GemmParams& prm);
// Whether a grouped GEMM of this size takes the split kernel (rows: of all experts).
bool split_gemm_ok(int k, int n, int experts, long rows, int cus);
enum class SplitShape { kBySize, kFourWaves, kEightWaves, kRows256 };
// Grouped (prm.sorted_route null) or chain form (no 256-row tiles). rows: of all
// experts (picks the tile shape); rows_per_expert sizes the grid only.
hipError_t split_grouped(const GemmParams& prm, long rows_per_expert, long rows, int cus, SplitShape shape,
                         hipStream_t stream);

}  // namespace rr::kern
