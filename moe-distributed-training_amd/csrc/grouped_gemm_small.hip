// The grouped GEMM with tiles of 128 x 128, 4 waves, two workgroups per compute unit.
#define MOE_GEMM_TILE 128
#include "grouped_gemm_kernel.h"

int moe_launch_gemm_small_tile(const MoeGemmParams& p, int64_t R, hipStream_t stream) { return launch_epilogue(p, R, stream); }
