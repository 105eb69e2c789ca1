// The grouped GEMM with tiles of 128 x 128, 4 waves, two workgroups per compute unit.
#define MOE_GEMM_TILE 128
#include "grouped_gemm_kernel.h"

int moe_launch_gemm_small_tile(const MoeGemmParams& p, int64_t R, hipStream_t stream)
{
    if (p.K % BK != 0 || p.nslab > MOE_MAX_SLABS) return MOE_ERR_UNSUPPORTED;
    if (p.epi == MOE_EPI_STORE) return p.nn ? launch_variant<true, MOE_EPI_STORE>(p, R, stream) : launch_variant<false, MOE_EPI_STORE>(p, R, stream);
    if (p.epi == MOE_EPI_SWIGLU) return p.nn ? MOE_ERR_UNSUPPORTED : launch_variant<false, MOE_EPI_SWIGLU>(p, R, stream);
    if (p.epi == MOE_EPI_SWIGLU_FUSED) {
        if (p.nn || p.ncc != 1) return MOE_ERR_UNSUPPORTED;
        if (!p.CB[0] || !p.CCP[0] || !p.Y[0]) return MOE_ERR_BAD_ARG;
        return launch_variant<false, MOE_EPI_SWIGLU_FUSED>(p, R, stream);
    }
    if (p.epi == MOE_EPI_SWIGLU_BWD) return p.nn ? launch_variant<true, MOE_EPI_SWIGLU_BWD>(p, R, stream) : launch_variant<false, MOE_EPI_SWIGLU_BWD>(p, R, stream);
    if (p.epi == MOE_EPI_SWIGLU_BWD_FUSED) {
        if (p.nn || p.nrc != 3 || p.ncc != 2) return MOE_ERR_UNSUPPORTED;
        for (int i = 0; i < 3; ++i) if (!p.RC[i] || !p.RCP[i] || (i < 2 && (!p.CB[i] || !p.CCP[i]))) return MOE_ERR_BAD_ARG;
        return launch_variant<false, MOE_EPI_SWIGLU_BWD_FUSED>(p, R, stream);
    }
    return MOE_ERR_BAD_ARG;
}
