// Tiled fp32 GEMM, 64 x 64 workgroup tile of four groups of 2 x 2 wavefronts that share its reduction (gemm_fast.h,
// finish_groups): products with too few tiles to fill the GPU.
#include "gemm_fast.h"

namespace thgpu {

int gemm_fast_64x64k4(const GemmArgs &g, int la, int lb, bool red, hipStream_t s) {
    return gemm_fast_dispatch<64, 64, 2, 2, 4>(g, la, lb, red, s);
}

}  // namespace thgpu
