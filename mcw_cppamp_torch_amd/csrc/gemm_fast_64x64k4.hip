// Tiled fp32 GEMM, 64 x 64 workgroup tile of four groups of 2 x 2 wavefronts that share its reduction (gemm_fast.h,
// finish_groups): products with too few tiles to fill the GPU.
#include "gemm_fast.h"

namespace thgpu {

int gemm_fast_64x64k4(const GemmArgs &g, int la, int lb, bool red, hipStream_t s) {
    return gemm_fast_dispatch<64, 64, 2, 2, 4>(g, la, lb, red, s);
}

bool gemm_fast_64x64k4_pairs(int la, int lb, bool red, int la2, int lb2, bool red2) {
    return la == LD_RC_VEC && lb == LD_XC_GATHER && !red && la2 == LD_RC_VEC &&
           (lb2 == LD_RC_GATHER || lb2 == LD_RC_GATHER_VEC) && red2;
}

int gemm_fast_64x64k4_pair(const GemmArgs &a, const GemmArgs &b, int lb2, hipStream_t s) {
    auto kernel = lb2 == LD_RC_GATHER_VEC ? gemm_pair_kernel<LD_RC_VEC, LD_XC_GATHER, false, LD_RC_VEC, LD_RC_GATHER_VEC, true>
                                          : gemm_pair_kernel<LD_RC_VEC, LD_XC_GATHER, false, LD_RC_VEC, LD_RC_GATHER, true>;
    hipLaunchKernelGGL(kernel, dim3(a.total + b.total), dim3(1024), 0, s, a, b);
    return 0;
}

}  // namespace thgpu
