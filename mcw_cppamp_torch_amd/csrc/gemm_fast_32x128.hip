// Tiled fp32 GEMM, 32 x 128 workgroup tile (1 x 4 wavefronts, each 32 x 32): products of at most 32 rows, of which a
// 64-row tile would multiply half for nothing.  First operand along r only (its 128 128-bit loads per step are made by
// the first two wavefronts).
#include "gemm_fast.h"

namespace thgpu {

int gemm_fast_32x128(const GemmArgs &g, int la, int lb, bool red, hipStream_t s) {
    if (la != LD_RC_VEC) return fail("gemm: the 32-row tiles take a first operand contiguous along r");
    if (lb == LD_RC_VEC)
        return red ? gemm_fast_go<32, 128, 1, 4, LD_RC_VEC, LD_RC_VEC, true>(g, s)
                   : gemm_fast_go<32, 128, 1, 4, LD_RC_VEC, LD_RC_VEC, false>(g, s);
    if (lb == LD_RC_GATHER && red) return gemm_fast_go<32, 128, 1, 4, LD_RC_VEC, LD_RC_GATHER, true>(g, s);
    if (lb == LD_RC_GATHER_VEC && red) return gemm_fast_go<32, 128, 1, 4, LD_RC_VEC, LD_RC_GATHER_VEC, true>(g, s);
    if (lb == LD_XC_GATHER && !red) return gemm_fast_go<32, 128, 1, 4, LD_RC_VEC, LD_XC_GATHER, false>(g, s);
    if (lb == LD_XC_SCALAR && !red) return gemm_fast_go<32, 128, 1, 4, LD_RC_VEC, LD_XC_SCALAR, false>(g, s);
    return fail("gemm: unknown loader combination (%d, %d)", la, lb);
}

}  // namespace thgpu
