// Tiled fp32 GEMM, 64 x 64 workgroup tile (2 x 2 wavefronts).
#include "gemm_fast.h"

#include <type_traits>

namespace thgpu {

int gemm_fast_64x64(const GemmArgs &g, int la, int lb, bool red, hipStream_t s) {
    return gemm_fast_dispatch<64, 64, 2, 2>(g, la, lb, red, s);
}

// Summing in two levels, for gathered gradInput products whose single long sum would be rounded more than the short ones that
// col2im adds up (GemmProblem::max_roundings).  A kernel of its own: with one more block of sums (93 -> 117 registers) four workgroups run on
// a CU where five did, which costs the other products of this tile 1 to 3 %.  134 planes from 495 indices (3x3, 57 images 19x19): 1.10e-7 -> 7.7e-8
// from 64 bits (columns 7.7e-8), 49.6 -> 50.1 us.
int gemm_fast_64x64f(const GemmArgs &g, int la, int lb, bool red, hipStream_t s) {
    if (la != LD_RC_VEC || lb != LD_XC_GATHER || red) return fail("gemm: the tile that sums in two levels gathers");
    return gemm_fast_go<64, 64, 2, 2, LD_RC_VEC, LD_XC_GATHER, false, 1, true>(g, s);
}

}  // namespace thgpu
