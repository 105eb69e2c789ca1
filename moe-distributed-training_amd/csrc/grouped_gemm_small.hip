// The grouped GEMM with tiles of 128 x 128, 4 waves, two workgroups per compute unit.
#define MOE_GEMM_TILE 128
#include "grouped_gemm_kernel.h"

int moe_launch_gemm_small_tile(const MoeGemmParams& p, int64_t R, hipStream_t stream) { return launch_epilogue(p, R, stream); }
int64_t moe_gemm_small_plan_blocks(int64_t R, int E, int64_t N, int pair) { return plan_blocks(R, E, N, pair); }
int moe_launch_gemm_small_plan(const void* offsets, int off64, int E, int64_t R, int64_t K, int64_t N, int pair, int nseg, int* out, hipStream_t stream)
{
    return launch_plan(offsets, off64, E, R, K, N, pair, nseg, out, stream);
}
