// The tiled fp32 GEMM kernel (see gemm_mfma.h for the problem statement): fp32 operands, fp32 sums and results, with the
// products formed on the bf16 matrix instructions.
//
// Every operand element is split into three bf16 parts, x = h + m + l: h is x rounded to nearest, m the
// remainder rounded, l what is left (8 + 8 + 8 significant bits hold the 24 of an fp32 number; without loss for zero
// and from 2^-110 up, see below).  A product a*b is the sum of the part products that matter in fp32,
// h*h + (h*m + m*h) + (h*l + m*m + l*h), each exact in the fp32 accumulator's
// input; the three dropped ones are below 2^-24 of the product together, and of either sign.  That is six
// v_mfma_f32_32x32x16_bf16 where eight v_mfma_f32_32x32x2_f32 of twice the cycles each stood: 2.7 times the matrix
// rate (dense bf16 runs at 16 times the fp32 rate).
//
// How the sums are rounded.  The bf16 instruction adds its sixteen products to the accumulator in two groups of eight, each
// rounded to nearest, after what lies far below the larger addend (2^-26 to 2^-32 of it, by which side is the
// smaller) has been cut towards minus infinity.  Left to run along the whole reduction, as in the fp32 kernel, that is
// twelve roundings of the full sum per sixteen indices (a sixth more error than before where half of an operand is zero,
// as behind a ReLU) and a mean error that grows with the reduction: -2.3e-7 of a result's standard deviation at 4608
// indices.  Sums over many results keep such a mean and pass it on: bias gradients of the AlexNet-style stack were 10
// times as far from 64 bits as with the fp32 instructions.  So
//   * the six products of one step (16 indices) are summed from zero, the small ones first, and the sum is added to the
//     accumulator by 16 vector additions: one rounding of the full sum per step;
//   * the sign of the product alternates: the first operand is negated in odd steps (its sum is then subtracted; free), the
//     second in odd columns (one v_xor_b32 per element), whose accumulators hold the negated result.  What the instruction
//     cuts pushes one step up and the next one down, one column up and its neighbour down.
// Error against 64 bits now: root mean square 0.25 to 0.6 of the fp32 instructions' from 64 indices up (uniform operands,
// half of one zero, positive: 0.26, 0.36 and 0.6 at 4608, 1024 and 576 indices), no mean error to be seen (below 2e-10);
// gradients of the AlexNet-style stack 2e-7 (fp32 instructions 3e-7 to 5e-7).  The additions cost a tenth: AlexNet-style step
// 3.2 -> 3.5 ms, VGG-A step 15.8 -> 17.0 ms, 64 -> 128 planes 9x9 9.1 -> 10.0 ms for the three passes.
//
// Against the fp32-instruction kernel that stood here (uniform random operands): AlexNet-style step at batch 128
// 4.51 -> 3.5 ms, 9x9 layer 13.2 -> 10.0 ms.  What bounds it is power and, with the additions, the vector unit: see the
// efficiency figures in gemm_dispatch.hip.
//
// What the split cannot hold is multiplied in fp32 instead, with v_mfma_f32_32x32x2_f32 (recompute):
//   * An operand below 2^-110 in magnitude can have bits under the smallest bf16 step, 2^-133, and then comes out short by
//     up to 2^-134.  Against a large partner that reaches a result of ordinary size, so it is found at the operand: what
//     l has to hold is a bf16 number exactly when the low half of its fp32 word is zero, and every thread collects these
//     words (one v_or3_b32 per two elements: AlexNet-style step 3.20 -> 3.24 ms, 64 -> 128 planes 9x9 9.1 -> 9.4 ms for the
//     three passes).  A workgroup that met a non-zero one multiplies its tile again.
//     (Conversion, subtraction and the matrix instruction keep denormals on gfx950, so nothing else is lost.)
//   * An operand that is infinite, NaN or so large that h rounds to infinity leaves an infinity or NaN in every
//     accumulator it reaches, and a product sum that falls below the normal numbers leaves a denormal: a wavefront
//     that finds one of these among its outputs computes them again.
//
// Structure
//   * A workgroup of WGM x WGN wavefronts owns a BM x BN tile of C, each
//     wavefront TM x TN blocks of 32x32 outputs, one accumulator (16 registers per lane) per block.
//   * No bounds checks and no branches around loads.  A tile at the lower/right
//     edge is shifted back so that it lies inside the matrix and stores only the
//     rows/columns no other tile owns; a reduction step that would run past R is
//     shifted back to end at R and the part the previous step already covered
//     is zeroed on its way to LDS.  Needs R >= 16 and, on sides longer than GEMM_SHORT_TILE, M >= BM and J >= BN.  A matrix
//     with fewer rows (columns) than a short side of the tile loads its last one in place of the missing ones and stores
//     only its own.
//   * The split is made once per element and workgroup, on the way from registers to LDS.  LDS holds the parts of both
//     operand tiles as [part][octet][x] units of eight bf16 (x the free index, octet = r/8): lane (x, h) of a wavefront
//     fetches its MFMA operand, r = 8h .. 8h+7 of row x, with one 128-bit read, consecutive lanes from
//     consecutive units.  The octet planes are 64 bytes longer than their rows need: LDS writes go to 32 banks (128 bytes),
//     and of sixteen lanes that write 64 bits each, four to a row, half then fall on each 64 bytes of them.  (With 128 bytes
//     both halves fell on the same banks: 95 % conflict cycles with both operands along r, 50 - 65 % with one, none now.
//     VGG-A step 2.5 % faster, 64 -> 128 planes 9x9 1 to 4 %; within the 2 % by which
//     cards differ on the AlexNet-style step.)
//   * LDS is double buffered and the global loads run one step further ahead: while step s is multiplied, the
//     registers hold step s+1, which is split and written to the other buffer in slices between the MFMAs, and every
//     register is refilled for step s+2 as soon as it has been split: one barrier per reduction step, and a load has a
//     whole step to arrive.
//   * Operands are fetched with buffer loads (descriptor and offsets in scalar registers, a constant lane offset), and
//     the loop is unrolled by two so that the LDS buffer folds into the offset field of the LDS instructions: the only
//     vector instructions of the loop are the split's (12 or, for the second operand, 14 per two elements) and the additions.
//   * The MFMAs go block by block.  The parts of the tile's shorter side stay in registers for the step; those of the longer
//     one are read from LDS a block row ahead, or just before their use where registers are short.
#pragma once

#include <type_traits>
#include <utility>

#include "gemm_mfma.h"

namespace thgpu {

// Loader kind used inside the kernel only: an x-contiguous first operand whose row count the thread
// count does not divide (192 rows, 256 threads).  Wavefront w takes r = 4w .. 4w+3 of every block of
// 64 consecutive rows; lanes run along the rows.
constexpr int LD_XC_BLOCK = 3;

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

// Bytes of one octet plane of an X-row operand tile, of one part of it, and of the whole tile.
template <int X>
struct PartTile {
    static constexpr int kOctet = X * 16 + 64;
    static constexpr int kPart = 2 * kOctet;
    static constexpr int kBytes = 3 * kPart;
};

// The three parts of two elements, two bf16 to a word.  `lost` collects the remainders that l rounds: a set bit in its low
// half says that some element was not held in full.
__device__ __forceinline__ void split_pair(float x0, float x1, unsigned &h, unsigned &m, unsigned &l, unsigned &lost) {
    auto round2 = [](float a, float b) {
        return __builtin_bit_cast(unsigned, __builtin_convertvector((floatx2){a, b}, bf16x2));
    };
    auto low = [](unsigned p) { return __builtin_bit_cast(float, p << 16); };
    auto high = [](unsigned p) { return __builtin_bit_cast(float, p & 0xffff0000u); };
    h = round2(x0, x1);
    const float r0 = x0 - low(h), r1 = x1 - high(h);
    m = round2(r0, r1);
    const float s0 = r0 - low(m), s1 = r1 - high(m);
    l = round2(s0, s1);
    // (written out: from the operators the compiler gathers the words of several pairs before it combines them, and spills)
    asm("v_or3_b32 %0, %0, %1, %2" : "+v"(lost) : "v"(s0), "v"(s1));
}

// f(0), f(1), ... with the index as a compile-time constant.
template <typename F, int... I>
__device__ __forceinline__ void for_each_index(F f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}

// Wavefronts per SIMD the register allocation must leave room for: the accumulators take (BM/WGM)*(BN/WGN)/64 registers
// of the 512 a lane has, and no more workgroups run on a CU than its 160 KB of LDS hold tile buffers for (four wavefronts
// each, one to a SIMD).
template <int BM, int BN, int WGM, int WGN>
constexpr int gemm_min_waves() {
    constexpr int by_lds = 160 * 1024 / (2 * (PartTile<BM>::kBytes + PartTile<BN>::kBytes));
    return (BM / WGM) * (BN / WGN) / 64 >= 96 || by_lds < 3 ? 2 : 3;
}

// The end of a workgroup of KG groups, each of which holds the sum of its own steps for the whole 64 x 64 tile: the groups'
// sums meet in LDS and are added in the order of the groups, a thread taking the four outputs of one register quad of one
// wavefront's block (and `rowsum`, the row sums of the first operand, likewise).
//
// What it is for: a step of the 64 x 64 tile has a latency of 0.4 to 0.6 us (its six products in a row, the split, LDS and
// a barrier), which a CU with one or two workgroups does not hide.  Four steps at once take as long, in the same LDS
// and registers that four workgroups of a quarter of the reduction would have, but without the partial sums, or with a
// quarter of them: 3x3 layers of one and three 13x13 images 18.0 -> 17.4 and 23.3 -> 21.4 us with their split reductions
// (27 -> 18 and 8 -> 5 parts), 50 images of 32 -> 64 planes 16x16 18.5 -> 16.0, their gradWeight 22.5 -> 19.0.
// Finishing a reduction that is split over workgroups here as well, in the one that arrives last, was tried and taken back:
// stores completed past the XCD's cache, a count and loads past it took the 4 us of the launch they replaced (256 x 169 over
// 3456: 13.7 + 4, 18 to 20 us), and twice that with agent-scope fences.
template <int BM, int BN, int WGN, bool RED, int KG>
__device__ __forceinline__ void finish_groups(const GemmArgs &g, char *lds_a, char *lds_b, const floatx16 &acc, float rowsum,
                                              bool rs_on, int group, int wave, int lane, unsigned tj, unsigned split, int i0, int j0, int own_i0,
                                              int own_j0) {
    static_assert(BM == 64 && BN == 64 && WGN == 2 && KG == 4, "sixteen wavefronts, sixteen quads of registers");
    const int thread = threadIdx.x, half = lane >> 5, l32 = lane & 31;
    // three groups' sums over the first operand's tiles, the last one's and the row sums over the second's
    auto frag = [&](int k) { return reinterpret_cast<floatx4 *>(k < KG - 1 ? lds_a + k * (BM * BN * 4) : lds_b); };
    float *const rows = reinterpret_cast<float *>(lds_b + BM * BN * 4);
    static_assert((KG - 1) * BM * BN * 4 <= KG * 2 * PartTile<BM>::kBytes, "LDS of the first operand");
    static_assert(BM * BN * 4 + KG * BM * 4 <= KG * 2 * PartTile<BN>::kBytes, "LDS of the second operand");
    __syncthreads();  // the flags of lost bits have been read
#pragma unroll
    for (int q = 0; q < 4; ++q)
        frag(group)[(wave * 4 + q) * 64 + lane] = (floatx4){acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    if (RED && rs_on) {
        float total = rowsum + __shfl_xor(rowsum, 1);  // four lanes hold the quarters of a row
        total += __shfl_xor(total, 2);
        if ((lane & 3) == 0) rows[group * BM + wave * 16 + (lane >> 2)] = total;
    }
    __syncthreads();
    const int of = thread >> 8, quad = (thread >> 6) & 3;  // whose outputs the thread takes over
    floatx4 sum = frag(0)[(of * 4 + quad) * 64 + lane];
#pragma unroll
    for (int k = 1; k < KG; ++k) sum += frag(k)[(of * 4 + quad) * 64 + lane];
    if (RED && rs_on && thread < BM) {
        const int i = i0 + thread;
        if (i >= own_i0 && i < g.M)
            g.rowsum_ws[(long)i * g.nsplit * g.tilesJ + (long)split * g.tilesJ + tj] =
                ((rows[thread] + rows[BM + thread]) + rows[2 * BM + thread]) + rows[3 * BM + thread];
    }

    // Four rows of one column.
    const int j = j0 + (of % WGN) * 32 + l32, i_first = i0 + (of / WGN) * 32 + 8 * quad + 4 * half;
    if (j < own_j0 || j >= g.J) return;
    const float sign = l32 & 1 ? -1.0f : 1.0f;  // odd columns hold the negated sum
    if (g.nsplit > 1) {
        float *const ws = g.ws + (long)split * g.M * g.J + j;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (i_first + e >= own_i0 && i_first + e < g.M) ws[(long)(i_first + e) * g.J] = sum[e] * sign;
        return;
    }
    const float alpha = sign * g.alpha;
    unsigned im, n, y, x;
    g.divN.divmod((unsigned)j, im, n);
    g.divCW.divmod(n, y, x);
    if (g.scatter) {
        const int hy = (int)y * g.scat_sH - g.scat_pH, wx = (int)x * g.scat_sW - g.scat_pW;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = i_first + e;
            unsigned c, rem, ph, pw;
            g.divScatS.divmod((unsigned)i, c, rem);
            g.divScatW.divmod(rem, ph, pw);
            const int h = hy + (int)ph, w = wx + (int)pw;
            if (i < own_i0 || i >= g.scat_rows || h < 0 || h >= g.scat_H || w < 0 || w >= g.scat_W) continue;
            const long off = (long)im * g.bsC + ((long)c * g.scat_H + h) * g.scat_W + w;
            float val = sum[e] * alpha + 0.0f;
            if (g.mask) val = g.mask[off] > g.mask_threshold ? val : 0.0f;
            g.C[off] = val;
        }
        return;
    }
    const bool per_image = !RED && (g.N != g.J || g.c_pitch != 0 || g.mask_pitch != 0 || g.C2 != nullptr);
    const long col = !per_image ? (long)j : (long)im * g.bsC + (g.c_pitch ? (long)y * g.c_pitch + x : (long)n);
    const long mcol = !per_image ? (long)j : (long)im * g.mask_bsC + (g.mask_pitch ? (long)y * g.mask_pitch + x : (long)n);
    const long tcol = (long)im * g.c2_bsC + (long)y * g.c2_pitch + x;
    const float col_bias = g.bias_col ? g.bias_col[j] : 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int i = i_first + e;
        if (i < own_i0 || i >= g.M) continue;
        float *const c = g.C + (long)i * g.sC + col;
        float val = sum[e] * alpha + ((g.bias ? g.bias[i] : 0.0f) + col_bias);
        if (g.beta != 0.0f) val += g.beta * *c;
        if (g.act) val = val > g.act_threshold ? val : g.act_value;
        if (g.mask) val = g.mask[(long)i * g.mask_sC + mcol] > g.mask_threshold ? val : 0.0f;
        *c = val;
        if (!RED && g.C2) g.C2[(long)i * g.c2_sC + tcol] = val;
    }
}

// One workgroup of a product; As and Bs hold KG pairs of operand tiles.  FOLD: every g.fold_steps steps (an even number) a
// wavefront's sum goes to a second one and starts over (gemm_roundings).
template <int BM, int BN, int WGM, int WGN, int LA, int LB, bool RED, int KG, bool FOLD = false>
__device__ __forceinline__ void gemm_fast_tile(const GemmArgs &g, const unsigned block, char *const As, char *const Bs) {
    constexpr int NT = WGM * WGN * 64;  // threads of a group: the whole workgroup unless KG > 1
    constexpr int BK = GEMM_BK;
    constexpr int TM = BM / WGM / 32, TN = BN / WGN / 32;
    // A first operand along r whose 128-bit loads the threads do not divide (96 rows: 384 loads, 256 threads): the
    // last round of loads is made by the leading wavefronts only (a uniform branch; wavefront w loads rows
    // 16w .. 16w+15 of every 64).
    constexpr bool PART_A = LA == LD_RC_VEC && (BM * BK) % (NT * 4) != 0;
    constexpr int NA = PART_A ? (BM * BK + NT * 4 - 1) / (NT * 4) * 4 : BM * BK / NT, NB = BN * BK / NT;
    static_assert(BK == 16, "two octets of reduction indices per step");
    static_assert(!PART_A || (NT == 256 && BM % 16 == 0), "partial loader shape");
    static_assert(BM % (WGM * 32) == 0 && BN % (WGN * 32) == 0, "wave tile must be whole 32x32 blocks");
    static_assert(NT % 16 == 0 && NA >= 4 && NB >= 4 && NA % 4 == 0 && NB % 4 == 0, "loader shape");
    // The kind the A loader really uses: x-contiguous with 192 rows goes block-wise.
    constexpr int KA = (LA == LD_XC_SCALAR && NT % BM != 0) ? LD_XC_BLOCK : LA;
    static_assert(KA != LD_XC_BLOCK || (NT == 256 && BM % 64 == 0 && NA == BM / 16), "block loader shape");
    static_assert((LB != LD_XC_SCALAR && LB != LD_XC_GATHER) || NT % BN == 0,
                  "x-contiguous loaders give every thread one row/column");
    static_assert(LB != LD_XC_GATHER || BN % 64 == 0, "a wavefront of the gathering loader shares its reduction indices");
    static_assert(LA == LD_RC_VEC || LA == LD_XC_SCALAR, "only the second operand is gathered");
    // The second operand gathered with four lanes to a column (element (r, x) at rowtab[r] + coltab[x] either way).
    constexpr bool RG = LB == LD_RC_GATHER || LB == LD_RC_GATHER_VEC;
    constexpr bool GATHER = LB == LD_XC_GATHER || RG;
    static_assert(!RG || (RED && NT == 256), "lanes along the reduction: reduction batching only");
    static_assert(!RED || (LA == LD_RC_VEC && (LB == LD_RC_VEC || RG)), "reduction batching needs operands loaded along r");
    constexpr bool SHORT_M = BM <= GEMM_SHORT_TILE, SHORT_J = BN <= GEMM_SHORT_TILE;
    static_assert(!SHORT_M || NT / 4 >= BM, "one round of loads along r covers the rows of a short tile");
    static_assert(!SHORT_J || NT / 4 >= BN, "and its columns");

    using TileA = PartTile<BM>;
    using TileB = PartTile<BN>;
    const int group = KG > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / NT) : 0;
    const int tid = KG > 1 ? threadIdx.x % NT : threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // scalar: row bases stay uniform
    const int wm = wave / WGN, wn = wave % WGN;
    const int half = lane >> 5, l32 = lane & 31;

    // ---- which tile, which part of the reduction --------------------------------
    unsigned pid = xcd_remap(block, g.total);
    unsigned ti, tj, split, rest;
    g.divTilesM.divmod(pid, rest, ti);
    g.divTilesJ.divmod(rest, split, tj);
    const int own_i0 = (int)ti * BM, own_j0 = (int)tj * BN;
    int i0 = own_i0 + BM <= g.M ? own_i0 : g.M - BM;  // shifted back at the edge
    int j0 = own_j0 + BN <= g.J ? own_j0 : g.J - BN;
    // A matrix with fewer rows or columns than the tile: its last row or column is loaded in place of the missing ones.
    if (SHORT_M && g.M < BM) i0 = 0;
    if (SHORT_J && g.J < BN) j0 = 0;
    auto row_at = [&](int i) { return SHORT_M && i >= g.M ? g.M - 1 : i; };
    auto col_at = [&](int j) { return SHORT_J && j >= g.J ? g.J - 1 : j; };

    int step = (int)split * g.steps_per_split;
    int step_end = step + g.steps_per_split;
    if (step_end > g.steps_total) step_end = g.steps_total;
    int rounds = 0;  // loop iterations of the longest group
    if constexpr (KG > 1) {
        rounds = (step_end - step + KG - 1) / KG;
        step += group * rounds;
        if (step_end > step + rounds) step_end = step + rounds;
        if (step_end < step) step_end = step;
    }
    const int nsteps = step_end - step;
    int ld_img = 0, ld_r0 = step * BK;
    if (RED) {
        unsigned im, st;
        g.divSpi.divmod((unsigned)step, im, st);
        ld_img = (int)im;
        ld_r0 = (int)st * BK;
    }

    // ---- loader set-up -------------------------------------------------------------
    // Thread -> (x, r) of its first element inside an operand tile:
    //   LD_RC_VEC     x = tid/4 (+64 per load), r = 4*(tid%4) .. +3   (one 128-bit load each)
    //   LD_XC_SCALAR  x = tid % X, r = (tid / X) * CNT .. + CNT-1     (CNT loads down the column)
    //   LD_XC_BLOCK   x = lane (+64 per block of rows), r = 4*wave .. +3
    // A load address is a wave-uniform base (tile, image, step, load number: all
    // scalar) plus a per-thread byte offset that never changes, so the loop
    // spends no vector ALU work on addressing.
    int a_x, a_r, b_x, b_r;
    unsigned voffA, voffB;
    const char *tileA, *tileB;
    if (KA == LD_XC_BLOCK) {
        a_x = lane;
        a_r = 4 * wave;
        voffA = (unsigned)(((long)a_r * g.sA + a_x) * 4);
        tileA = reinterpret_cast<const char *>(g.A + i0);
    } else if (LA == LD_XC_SCALAR) {
        a_x = tid % BM;
        a_r = (tid / BM) * NA;
        voffA = (unsigned)(((long)a_r * g.sA + (row_at(i0 + a_x) - i0)) * 4);
        tileA = reinterpret_cast<const char *>(g.A + i0);
    } else {
        a_x = tid >> 2;
        a_r = (tid & 3) * 4;
        voffA = (unsigned)(((long)(row_at(i0 + a_x) - i0) * g.sA + a_r) * 4);
        tileA = reinterpret_cast<const char *>(g.A + (long)i0 * g.sA);
    }
    // Lanes along r: the column offsets in bytes of the thread's column of every 64.
    unsigned coffB[RG ? NB / 4 : 1];
    if (RG) {
        b_x = tid >> 2;
        b_r = (tid & 3) * 4;
        voffB = 0;
#pragma unroll
        for (int q = 0; q < (RG ? NB / 4 : 1); ++q) coffB[q] = (unsigned)g.coltab[col_at(j0 + b_x + q * (NT / 4))] * 4u;
        tileB = reinterpret_cast<const char *>(g.B);
    } else if (LB == LD_XC_GATHER) {
        b_x = tid % BN;
        b_r = (wave * 64 / BN) * NB;  // = (tid / BN) * NB, kept uniform: the row offsets are scalar loads
        unsigned img0, n0, img, n;
        g.divN.divmod((unsigned)j0, img0, n0);
        g.divN.divmod((unsigned)col_at(j0 + b_x), img, n);
        voffB = (unsigned)(((long)(img - img0) * g.bsB + g.coltab[n]) * 4);
        tileB = reinterpret_cast<const char *>(g.B + (long)img0 * g.bsB);
    } else if (LB == LD_XC_SCALAR) {
        b_x = tid % BN;
        b_r = (tid / BN) * NB;
        unsigned img0, n0, img, n;
        g.divN.divmod((unsigned)j0, img0, n0);
        g.divN.divmod((unsigned)col_at(j0 + b_x), img, n);
        voffB = (unsigned)(((long)b_r * g.sB + (long)(img - img0) * g.bsB + n) * 4);
        tileB = reinterpret_cast<const char *>(g.B + (long)img0 * g.bsB);
    } else {
        b_x = tid >> 2;
        b_r = (tid & 3) * 4;
        voffB = (unsigned)(((long)(col_at(j0 + b_x) - j0) * g.sB + b_r) * 4);
        tileB = reinterpret_cast<const char *>(g.B + (long)j0 * g.sB);
    }
    constexpr int UA = LA == LD_RC_VEC ? NA / 4 : NA;  // load instructions per step and operand
    constexpr int UB = LB == LD_RC_VEC || LB == LD_RC_GATHER_VEC ? NB / 4 : NB;

    floatx16 acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;

    // Row sums of the first operand (GemmProblem::rowsum), reduction batching only.  The column tiles of a row of
    // tiles all load the same first-operand tiles, so they share the work: the workgroup of column tile tj sums the
    // steps whose index is tj modulo the number of column tiles, from the registers the loads arrive in (fp32, before the
    // split; thread t holds four elements of row t/4 of every 64).  A handful of vector adds every tilesJ-th step; the
    // partial sums go to rowsum_ws[row][split * tilesJ + tj].
    constexpr int RS = RED ? NA / 4 : 1;
    float bsum[RS];
#pragma unroll
    for (int q = 0; q < RS; ++q) bsum[q] = 0.0f;
    const bool rs_on = RED && g.rowsum_ws != nullptr;
    int rs_next = 0;
    if (rs_on) rs_next = (int)(((unsigned)tj + g.tilesJ - (unsigned)step % g.tilesJ) % g.tilesJ);

    float ra[NA], rb[NB];
    auto a_unit_live = [&](int u) { return !PART_A || u * (NT / 4) + 16 * wave < BM; };
    if (PART_A) {
#pragma unroll
        for (int q = 0; q < NA; ++q) ra[q] = 0.0f;
    }
    // Gathered B: float offsets of the rows of the step being loaded (uniform), and of the step after it.  The
    // latter are fetched (scalar loads) in the middle of a step, a whole step before they turn into addresses,
    // so that no step starts by waiting for its row offsets.
    // (With lanes along r each lane holds the offsets of its own four r, or of the first of them.)
    constexpr int NROW = LB == LD_XC_GATHER ? NB : LB == LD_RC_GATHER ? 4 : 1;
    int roff[NROW], roff_nx[NROW];

    // Load number u of an operand for the step whose uniform base is `base`.  Buffer loads: the address is a
    // descriptor in scalar registers (the step's base) plus a scalar offset (which load) plus the lane's constant
    // 32-bit offset, so the loop spends no vector ALU instruction on addressing.
    typedef float float4v __attribute__((ext_vector_type(4)));
    auto descriptor = [](const char *base) {
        // raw buffer, no bounds (every offset below 2^32 passes), dword format
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(base), 0, -1, 0x00020000);
    };
    auto load_unit = [&](auto kind_tag, const char *base, long stride, unsigned voff, float *dst, int u) {
        constexpr int KIND = decltype(kind_tag)::value;
        const __amdgpu_buffer_rsrc_t rsrc = descriptor(base);
        const int st = (int)stride * 4;
        if (KIND == LD_RC_VEC) {
            const float4v v = __builtin_bit_cast(
                float4v, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)voff, u * (NT / 4) * st, 0));
            dst[u * 4 + 0] = v.x;
            dst[u * 4 + 1] = v.y;
            dst[u * 4 + 2] = v.z;
            dst[u * 4 + 3] = v.w;
        } else if (KIND == LD_RC_GATHER_VEC) {
            const float4v v = __builtin_bit_cast(
                float4v, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(coffB[u % (RG ? NB / 4 : 1)] + (unsigned)roff[0] * 4u), 0, 0));
            dst[u * 4 + 0] = v.x;
            dst[u * 4 + 1] = v.y;
            dst[u * 4 + 2] = v.z;
            dst[u * 4 + 3] = v.w;
        } else if (KIND == LD_RC_GATHER) {
            dst[u] = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(
                           rsrc, (int)(coffB[u / 4 % (RG ? NB / 4 : 1)] + (unsigned)roff[u % 4 % NROW] * 4u), 0, 0));
        } else {
            const int so = KIND == LD_XC_BLOCK    ? (u & 3) * st + (u >> 2) * 256
                           : KIND == LD_XC_GATHER ? roff[u % NROW] * 4
                                                  : u * st;
            dst[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)voff, so, 0));
        }
    };

    // Uniform bases of the step at (ld_img, ld_r0).  A step that would run past
    // R is moved back to end at R (every address stays inside the operand;
    // needs R >= BK); `shift` says how many of its leading reduction indices the
    // previous step already covered -- those are zeroed before they reach LDS.
    auto step_bases = [&](const char *&ga, const char *&gb, int &shift) {
        const int r0 = ld_r0 + BK <= g.R ? ld_r0 : g.R - BK;
        shift = ld_r0 - r0;
        ga = tileA + ((RED ? (long)ld_img * g.rbA : 0L) + (LA == LD_XC_SCALAR ? (long)r0 * g.sA : (long)r0)) * 4;
        if (GATHER) {
            gb = tileB + (RED ? (long)ld_img * g.rbB : 0L) * 4;
#pragma unroll
            for (int u = 0; u < NROW; ++u) roff[u] = roff_nx[u];
        } else {
            gb = tileB + ((RED ? (long)ld_img * g.rbB : 0L) + (LB == LD_XC_SCALAR ? (long)r0 * g.sB : (long)r0)) * 4;
        }
    };
    // Row offsets of the step whose reduction window starts at `pos` (moved back like the step itself).
    auto fetch_rows = [&](int pos) {
        if (GATHER) {
            const int r0 = pos + BK <= g.R ? pos : g.R - BK;
            const int *rt = g.rowtab + r0 + b_r;
#pragma unroll
            for (int u = 0; u < NROW; ++u) roff_nx[u] = rt[u];
        }
    };
    // Takes delivery of them (an empty statement that names the values keeps the compiler from postponing the
    // loads to the point of first use).
    auto pin_rows = [&]() {
        if (LB == LD_XC_GATHER) {
#pragma unroll
            for (int u = 0; u < NROW; ++u) {
                int t = __builtin_amdgcn_readfirstlane(roff_nx[u]);
                asm("" : "+s"(t));
                roff_nx[u] = t;
            }
        }
    };
    auto advance = [&]() {
        ld_r0 += BK;
        if (RED && ld_r0 >= g.R) {
            ld_r0 = 0;
            ++ld_img;
        }
    };
    // Zero the elements whose position inside the step window is below `shift`.
    auto mask_one = [&](auto kind_tag, int t_r, float *v, auto count_tag, int shift) {
        constexpr int KIND = decltype(kind_tag)::value;
        constexpr int CNT = decltype(count_tag)::value;
#pragma unroll
        for (int q = 0; q < CNT; ++q) {
            const int rel = (KIND == LD_XC_SCALAR || KIND == LD_XC_GATHER) ? t_r + q : t_r + (q & 3);
            v[q] = rel < shift ? 0.0f : v[q];
        }
    };
    auto mask_step = [&](int shift) {
        if (shift > 0) {  // uniform: only the last step of an image can be partial
            mask_one(std::integral_constant<int, KA>{}, a_r, ra, std::integral_constant<int, NA>{}, shift);
            mask_one(std::integral_constant<int, LB>{}, b_r, rb, std::integral_constant<int, NB>{}, shift);
        }
    };

    // Splits group number q of a thread's elements and writes the parts to LDS.  A group is eight elements of a row
    // where the loader gives a thread whole octets, otherwise four.
    constexpr int GA = (KA == LD_XC_SCALAR && NA % 8 == 0) ? 8 : 4;
    constexpr int GB = ((LB == LD_XC_SCALAR || LB == LD_XC_GATHER) && NB % 8 == 0) ? 8 : 4;
    char *const a_dst = As + group * (2 * TileA::kBytes) + (a_r >> 3) * TileA::kOctet + a_x * 16 + (a_r & 7) * 2;
    char *const b_dst = Bs + group * (2 * TileB::kBytes) + (b_r >> 3) * TileB::kOctet + b_x * 16 + (b_r & 7) * 2;
    unsigned lost = 0;  // see split_pair
    const unsigned odd_column = (unsigned)(b_x & 1) << 31;  // the sign of a thread's elements of the second operand
    auto stash_group = [&](auto kind_tag, auto group_tag, auto tile_tag, char *dst, const float *src, int q, auto sign) {
        constexpr int KIND = decltype(kind_tag)::value;
        constexpr int G = decltype(group_tag)::value;
        using Tile = decltype(tile_tag);
        // four-element groups lie in rows apart (four lanes to a row: NT/4 rows, LD_XC_BLOCK: the next 64 rows)
        const int off = G == 8 ? q * Tile::kOctet : (KIND == LD_XC_BLOCK ? q * 64 : q * (NT / 4)) * 16;
        unsigned p[3][G / 2];
#pragma unroll
        for (int e = 0; e < G / 2; ++e) split_pair(sign(src[q * G + 2 * e]), sign(src[q * G + 2 * e + 1]), p[0][e], p[1][e], p[2][e], lost);
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            if constexpr (G == 8)
                *reinterpret_cast<uintx4 *>(dst + off + t * Tile::kPart) = (uintx4){p[t][0], p[t][1], p[t][2], p[t][3]};
            else
                *reinterpret_cast<uintx2 *>(dst + off + t * Tile::kPart) = (uintx2){p[t][0], p[t][1]};
        }
    };
    static_assert(GA == 8 || KA != LD_XC_SCALAR || NA == 4, "an x-contiguous loader of four elements has one group");
    static_assert(GB == 8 || LB == LD_RC_VEC || RG || NB == 4, "an x-contiguous loader of four elements has one group");
    auto stash_a = [&](int buf, int q) {
        if (GA == 8 || a_unit_live(q))
            stash_group(std::integral_constant<int, KA>{}, std::integral_constant<int, GA>{}, TileA{},
                        a_dst + buf * TileA::kBytes, ra, q, [&](float x) { return buf ? -x : x; });
    };
    auto stash_b = [&](int buf, int q) {
        stash_group(std::integral_constant<int, LB>{}, std::integral_constant<int, GB>{}, TileB{},
                    b_dst + buf * TileB::kBytes, rb, q,
                    [&](float x) { return __builtin_bit_cast(float, __builtin_bit_cast(unsigned, x) ^ odd_column); });
    };
    constexpr int QA = NA / GA, QB = NB / GB;
    // The loads that refill group q.
    auto refill_a = [&](const char *base, int q) {
        constexpr int PER = UA / QA;
#pragma unroll
        for (int u = q * PER; u < (q + 1) * PER; ++u)
            if (a_unit_live(u)) load_unit(std::integral_constant<int, KA>{}, base, g.sA, voffA, ra, u);
    };
    auto refill_b = [&](const char *base, int q) {
        constexpr int PER = UB / QB;
#pragma unroll
        for (int u = q * PER; u < (q + 1) * PER; ++u) load_unit(std::integral_constant<int, LB>{}, base, g.sB, voffB, rb, u);
    };
    auto add_row_sums = [&]() {
        if constexpr (RED) {
#pragma unroll
            for (int q = 0; q < RS; ++q) bsum[q] += (ra[4 * q] + ra[4 * q + 1]) + (ra[4 * q + 2] + ra[4 * q + 3]);
        }
    };

    // ---- prologue: the first step to LDS, the second to registers ---------------------
    const char *ga = tileA, *gb = tileB;
    int shift = 0;
    if (nsteps > 0) {
        fetch_rows(ld_r0);
        step_bases(ga, gb, shift);
#pragma unroll
        for (int q = 0; q < QA; ++q) refill_a(ga, q);
#pragma unroll
        for (int q = 0; q < QB; ++q) refill_b(gb, q);
        advance();
        fetch_rows(ld_r0);
        mask_step(shift);
        if (rs_on && rs_next == 0) {
            add_row_sums();
            rs_next = (int)g.tilesJ;
        }
#pragma unroll
        for (int q = 0; q < QA; ++q) stash_a(0, q);
#pragma unroll
        for (int q = 0; q < QB; ++q) stash_b(0, q);
        if (nsteps > 1) {
            step_bases(ga, gb, shift);
#pragma unroll
            for (int q = 0; q < QA; ++q) refill_a(ga, q);
#pragma unroll
            for (int q = 0; q < QB; ++q) refill_b(gb, q);
            advance();
            fetch_rows(ld_r0);
        }
    }
    __syncthreads();

    // ---- main loop ----------------------------------------------------------------------
    // Step s multiplies from LDS buffer s&1, block by block; between the MFMAs the groups of
    // step s+1 are split and written to the other buffer and their registers refilled for step s+2.
    const char *const a_src = As + group * (2 * TileA::kBytes) + half * TileA::kOctet + (wm * (TM * 32) + l32) * 16;
    const char *const b_src = Bs + group * (2 * TileB::kBytes) + half * TileB::kOctet + (wn * (TN * 32) + l32) * 16;
    // Two sums in turn, so that the additions of one block run under the MFMAs of the next, where the registers hold both
    // (1 to 2 % on the 8-block tiles), and the parts of the longer side one block row ahead likewise.
    constexpr bool PING = !(TM == 2 && TN == 2 && WGN == 2) && !(TM * TN == 8 && LB == LD_RC_GATHER);
    constexpr int AHEAD = TM * TN == 8 || LB == LD_RC_GATHER ? 0 : 1;
    auto one_step = [&](auto buf_tag, int s) {
        constexpr int buf = decltype(buf_tag)::value;
        // The last step splits registers that nobody will read and the last two load from the previous addresses
        // (valid, cached) rather than branching around either.
        const bool more = s + 2 < nsteps;
        mask_step(shift);
        if (rs_on && s + 1 == rs_next && s + 1 < nsteps) {  // uniform
            add_row_sums();
            rs_next += (int)g.tilesJ;
        }
        if (more) step_bases(ga, gb, shift);

        if (RG) {  // vector loads: ahead of this step's refills, whose arrival nobody should wait for on their account
            int pos = ld_r0 + BK;
            if (pos >= g.R) pos = 0;
            fetch_rows(pos);
        }
        // Block by block; the parts of the tile's shorter side stay, those of the longer one are read a block row ahead.
        constexpr bool A_STAYS = TM <= TN;
        constexpr int STAY = A_STAYS ? TM : TN, PASS = A_STAYS ? TN : TM, BLOCKS = TM * TN;
        bf16x8 stay[STAY][3], pass[1 + AHEAD][3];
        auto read_a = [&](int a, int t) {
            return *reinterpret_cast<const bf16x8 *>(a_src + buf * TileA::kBytes + t * TileA::kPart + a * 512);
        };
        auto read_b = [&](int b, int t) {
            return *reinterpret_cast<const bf16x8 *>(b_src + buf * TileB::kBytes + t * TileB::kPart + b * 512);
        };
        auto read_pass = [&](int k) {
#pragma unroll
            for (int t = 2; t >= 0; --t) pass[k & AHEAD][t] = A_STAYS ? read_b(k, t) : read_a(k, t);
        };
#pragma unroll
        for (int t = 2; t >= 0; --t)
#pragma unroll
            for (int k = 0; k < STAY; ++k) stay[k][t] = A_STAYS ? read_a(k, t) : read_b(k, t);
        if (AHEAD) read_pass(0);
        floatx16 sum[PING ? 2 : 1];
        auto add_sum = [&](int block) {
            const int k = block / STAY, m = block % STAY;
            floatx16 &to = A_STAYS ? acc[m][k] : acc[k][m];
#pragma unroll
            for (int v = 0; v < 16; ++v) to[v] = buf ? to[v] - sum[PING ? block & 1 : 0][v] : to[v] + sum[PING ? block & 1 : 0][v];
            asm volatile("" : "+v"(to));  // here: left to itself the compiler moves the additions behind the step, sums and all
        };
        auto block_of = [&](auto block_tag) {
            constexpr int block = decltype(block_tag)::value;
            constexpr int k = block / STAY, m = block % STAY;
            if (m == 0 && k + AHEAD < PASS) read_pass(k + AHEAD);
            floatx16 part;
#pragma unroll
            for (int v = 0; v < 16; ++v) part[v] = 0.0f;
#pragma unroll
            for (int u = 0; u < 6; ++u) {
                // lh hl mm mh hm hh: the small ones first, while the sum is still small
                const int pa = u == 0 ? 2 : u == 2 || u == 3 ? 1 : 0;
                const int pb = u == 1 ? 2 : u == 2 || u == 4 ? 1 : 0;
                part = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A_STAYS ? stay[m][pa] : pass[k & AHEAD][pa],
                                                               A_STAYS ? pass[k & AHEAD][pb] : stay[m][pb], part, 0, 0, 0);
            }
            sum[PING ? block & 1 : 0] = part;
            if (PING && block > 0) add_sum(block - 1);
#pragma unroll
            for (int q = 0; q < QA; ++q)
                if (q * BLOCKS / (QA + QB) == block) {
                    stash_a(buf ^ 1, q);
                    refill_a(ga, q);
                }
#pragma unroll
            for (int q = 0; q < QB; ++q)
                if ((QA + q) * BLOCKS / (QA + QB) == block) {
                    stash_b(buf ^ 1, q);
                    refill_b(gb, q);
                }
            if (block == BLOCKS / 2 && !RG) {
                int pos = ld_r0 + BK;
                if (RED && pos >= g.R) pos = 0;
                fetch_rows(pos);
            }
            if (!RED && block == BLOCKS - 1) pin_rows();
            // One MFMA, then a few vector instructions under it (a 32x32x16 MFMA holds the matrix unit for 32 cycles, a vector
            // instruction issues in 4): 2 % over leaving them in clusters; 4, 6 and 8 measure alike.
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, 6, 0);
            }
            if (!PING || block == BLOCKS - 1) add_sum(block);
            __builtin_amdgcn_sched_barrier(0);
        };
        for_each_index(block_of, std::make_integer_sequence<int, BLOCKS>{});
        if (more) advance();
        else shift = 0;
        if (KG == 1) __syncthreads();
    };
    if constexpr (FOLD) {
        static_assert(KG == 1 && TM * TN == 1, "one more block of sums in the registers");
        floatx16 folded = {};
        for (int s = 0; s < nsteps;) {
            const int until = nsteps - s > g.fold_steps ? s + g.fold_steps : nsteps;
            do {
                one_step(std::integral_constant<int, 0>{}, s);
                if (s + 1 < nsteps) one_step(std::integral_constant<int, 1>{}, s + 1);
                s += 2;
            } while (s < until);
            folded += acc[0][0];
            acc[0][0] = (floatx16){};
        }
        acc[0][0] = folded;
    } else if constexpr (KG == 1) {
        for (int s = 0; s < nsteps; s += 2) {
            one_step(std::integral_constant<int, 0>{}, s);
            if (s + 1 < nsteps) one_step(std::integral_constant<int, 1>{}, s + 1);
        }
    } else {
        for (int s = 0; s < rounds; s += 2) {  // the last groups may have fewer steps, the barriers are everybody's
            if (s < nsteps) one_step(std::integral_constant<int, 0>{}, s);
            __syncthreads();
            if (s + 1 < nsteps) one_step(std::integral_constant<int, 1>{}, s + 1);
            __syncthreads();
        }
    }

    // ---- what the split could not hold -----------------------------------------------------
    // Did any thread's element lose bits?  (The operand tiles in LDS have been read: the loop ends with a barrier.)
    unsigned *const lost_of = reinterpret_cast<unsigned *>(As);
    const bool lost_here = __builtin_amdgcn_ballot_w64((lost & 0xffffu) != 0) != 0;
    if (lane == 0) lost_of[group * (NT / 64) + wave] = lost_here ? 1u : 0u;
    __syncthreads();
    unsigned lost_any = 0;
#pragma unroll
    for (int w = 0; w < KG * NT / 64; ++w) lost_any |= lost_of[w];
    // The wavefront's outputs in fp32, straight from the operands: eight reduction indices at a time, four to a lane half,
    // whose loads are in flight together.  (A step that would run past R is moved back as in the main loop.)
    const float column_sign = l32 & 1 ? -1.0f : 1.0f;  // of the accumulators
    auto recompute = [&]() {
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
            for (int b = 0; b < TN; ++b)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;
        struct __attribute__((packed, aligned(4))) Quad {
            float v[4];
        };
        const float *arow[TM], *bcol[TN];
#pragma unroll
        for (int a = 0; a < TM; ++a) {
            const long i = row_at(i0 + wm * (TM * 32) + a * 32 + l32);
            arow[a] = g.A + (LA == LD_XC_SCALAR ? i : i * g.sA);
        }
#pragma unroll
        for (int b = 0; b < TN; ++b) {
            const unsigned j = (unsigned)col_at(j0 + wn * (TN * 32) + b * 32 + l32);
            unsigned im = 0, n = j;
            if (!RED && LB != LD_RC_VEC) g.divN.divmod(j, im, n);
            bcol[b] = g.B + (GATHER               ? (long)im * g.bsB + g.coltab[n]
                             : LB == LD_XC_SCALAR ? (long)im * g.bsB + n
                                                  : (long)j * g.sB);
        }
#pragma unroll 1
        for (int st = step; st < step_end; ++st) {
            unsigned img = 0, w = (unsigned)st;
            if (RED) g.divSpi.divmod((unsigned)st, img, w);
            const int first = (int)w * BK, r0 = first + BK <= g.R ? first : g.R - BK;
            const long imA = RED ? (long)img * g.rbA : 0L, imB = RED ? (long)img * g.rbB : 0L;
#pragma unroll 1
            for (int c = 0; c < BK; c += 8) {
                const int r = r0 + c + 4 * half;  // the lane's r .. r+3
                float x[TM][4], y[TN][4];
#pragma unroll
                for (int a = 0; a < TM; ++a)
                    if (LA == LD_XC_SCALAR) {
#pragma unroll
                        for (int t = 0; t < 4; ++t) x[a][t] = arow[a][(long)(r + t) * g.sA];
                    } else {
                        const Quad q = *reinterpret_cast<const Quad *>(arow[a] + imA + r);
#pragma unroll
                        for (int t = 0; t < 4; ++t) x[a][t] = q.v[t];
                    }
                int off[4];
                if (GATHER) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) off[t] = g.rowtab[r + t];
                }
#pragma unroll
                for (int b = 0; b < TN; ++b)
                    if (LB == LD_RC_VEC) {
                        const Quad q = *reinterpret_cast<const Quad *>(bcol[b] + imB + r);
#pragma unroll
                        for (int t = 0; t < 4; ++t) y[b][t] = q.v[t];
                    } else {
#pragma unroll
                        for (int t = 0; t < 4; ++t) y[b][t] = bcol[b][imB + (GATHER ? (long)off[t] : (long)(r + t) * g.sB)];
                    }
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const bool covered = r + t < first;  // by the step before
#pragma unroll
                    for (int a = 0; a < TM; ++a) x[a][t] = covered ? 0.0f : x[a][t];
#pragma unroll
                    for (int b = 0; b < TN; ++b) y[b][t] = covered ? 0.0f : y[b][t] * column_sign;
#pragma unroll
                    for (int a = 0; a < TM; ++a)
#pragma unroll
                        for (int b = 0; b < TN; ++b)
                            acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[a][t], y[b][t], acc[a][b], 0, 0, 0);
                }
            }
        }
    };
    bool odd = lost_any != 0;
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) odd |= __builtin_amdgcn_classf(acc[a][b][v], 0x297);  // NaN, infinite, denormal
    if (__builtin_amdgcn_ballot_w64(odd)) recompute();

    // ---- groups ------------------------------------------------------------------------
    if constexpr (KG > 1) {
        finish_groups<BM, BN, WGN, RED, KG>(g, As, Bs, acc[0][0], bsum[0], rs_on, group, wave, lane, tj, split, i0, j0, own_i0, own_j0);
        return;
    }

    // ---- epilogue ----------------------------------------------------------------------
    // Accumulator register v of lane l holds D[8*(v/4) + 4*(l/32) + v%4][l%32].
    // A store address is a wave-uniform row base plus a constant per-lane byte
    // offset (column, image and the lane half's four rows), as for the loads.
    // MODE 0: partial sums to the workspace; 1: alpha*acc (+bias); 2: also + beta*C.
    // An edge tile: some rows or columns belong to its neighbour, or lie outside the matrix.
    const bool edge_tile = i0 != own_i0 || j0 != own_j0 || (SHORT_M && g.M < BM) || (SHORT_J && g.J < BN);
    auto write_out = [&](auto mode_tag, auto check_tag) {
        constexpr int MODE = decltype(mode_tag)::value;
        constexpr bool CHECK = decltype(check_tag)::value;
        const long row_bytes = (MODE == 0 ? (long)g.J : g.sC) * 4;
        char *const out0 = MODE == 0 ? reinterpret_cast<char *>(g.ws + (long)split * g.M * g.J)
                                     : reinterpret_cast<char *>(g.C);
        // Fused threshold / mask of the final value (uniform conditions; both off for partial sums).
        const float alpha = MODE != 0 ? column_sign * g.alpha : column_sign;  // (and + 0 makes a zero positive)
        const bool act = MODE != 0 && g.act != 0;
        const bool masked = MODE != 0 && g.mask != nullptr;
        const long mask_row_bytes = g.mask_sC * 4;
        unsigned img0 = 0, n0 = 0;
        // columns are (image, position) pairs, or positions of an image plane whose rows are kept apart
        const bool twin = MODE != 0 && !RED && g.C2 != nullptr;  // a second copy of the result (GemmProblem::C2)
        const long twin_row_bytes = g.c2_sC * 4;
        const bool per_image = MODE != 0 && !RED && (g.N != g.J || g.c_pitch != 0 || g.mask_pitch != 0 || twin);
        if (per_image) g.divN.divmod((unsigned)j0, img0, n0);
        char *const out = out0 + (per_image ? (long)img0 * g.bsC : (long)j0) * 4;
        const char *const msk = reinterpret_cast<const char *>(g.mask) + (per_image ? (long)img0 * g.mask_bsC : (long)j0) * 4;
        char *const out2 = reinterpret_cast<char *>(g.C2) + (long)img0 * g.c2_bsC * 4;
        // Per 32-column block of the wavefront: the lane's byte offset (into C, into the mask) and whether this tile
        // owns the column.
        unsigned voff[TN], mvoff[TN], tvoff[TN];
        bool own[TN];
        float col_bias[TN];
#pragma unroll
        for (int b = 0; b < TN; ++b) {
            const int jt = j0 + wn * (TN * 32) + b * 32 + l32;
            own[b] = jt >= own_j0 && (!SHORT_J || jt < g.J);  // else the neighbouring tile stores it, or there is no such column
            const int jg = CHECK ? col_at(jt) : jt;
            col_bias[b] = MODE != 0 && g.bias_col ? g.bias_col[jg] : 0.0f;
            long col = jg - j0, mcol = jg - j0, tcol = 0;
            if (per_image) {
                unsigned im, n, y, x;
                g.divN.divmod((unsigned)jg, im, n);
                g.divCW.divmod(n, y, x);
                col = (long)(im - img0) * g.bsC + (g.c_pitch ? (long)y * g.c_pitch + x : (long)n);
                mcol = (long)(im - img0) * g.mask_bsC + (g.mask_pitch ? (long)y * g.mask_pitch + x : (long)n);
                tcol = (long)(im - img0) * g.c2_bsC + (long)y * g.c2_pitch + x;
            }
            voff[b] = (unsigned)(col * 4 + 4 * half * row_bytes);
            mvoff[b] = (unsigned)(mcol * 4 + 4 * half * mask_row_bytes);
            tvoff[b] = (unsigned)(tcol * 4 + 4 * half * twin_row_bytes);
        }
        // Whether the lane's row ir + 4*half belongs to the tile above or lies below the matrix, of which an edge tile has only
        // one kind: a single comparison.
        const bool few_rows = SHORT_M && g.M < BM;
        const int edge_lane = few_rows ? -4 * half : 4 * half;
        auto not_ours = [&](int ir) { return edge_lane < (few_rows ? ir - g.M + 1 : own_i0 - ir); };
        // Rows outermost, the wavefront's column blocks innermost: the stores of one output row follow each other
        // directly, so a cache line that two neighbouring 128-byte segments share (rows are rarely 128-byte aligned)
        // is completed while it is still in L2 instead of going out to memory twice.
#pragma unroll
        for (int a = 0; a < TM; ++a) {
            const int iu = i0 + wm * (TM * 32) + a * 32;  // uniform
            float bias_v[16];
            if (MODE != 0 && g.bias) {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    bias_v[v] = CHECK && SHORT_M
                                    ? g.bias[row_at(iu + 8 * (v / 4) + (v % 4) + 4 * half)]
                                    : *reinterpret_cast<const float *>(
                                          reinterpret_cast<const char *>(g.bias + iu + 8 * (v / 4) + (v % 4)) + 16 * half);
            } else {
#pragma unroll
                for (int v = 0; v < 16; ++v) bias_v[v] = 0.0f;
            }
            // What C held, requested in batches of sixteen loads before the stores that need them.  A load per store, each
            // waited for, ran a 4096 x 9216 accumulation over 128 indices at 1.7 TB/s; one batch of all 16 * TN spilled
            // 60 to 300 registers (118 us, 2.6 TB/s; 96 us and 3.2 now, 4096 x 4096 77 -> 49 us).
            constexpr int ROWS = MODE == 2 && TN > 1 ? 16 / TN : 16;
            float held[MODE == 2 ? ROWS : 1][MODE == 2 ? TN : 1];
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                if (MODE == 2 && v % ROWS == 0) {
#pragma unroll
                    for (int q = 0; q < ROWS; ++q) {
                        const int ir = iu + 8 * ((v + q) / 4) + ((v + q) % 4);
#pragma unroll
                        for (int b = 0; b < TN; ++b)
                            held[MODE == 2 ? q : 0][MODE == 2 ? b : 0] =
                                !(CHECK && SHORT_M) || ir + 4 * half < g.M
                                    ? *reinterpret_cast<const float *>(out + (long)ir * row_bytes + voff[b])
                                    : 0.0f;
                    }
                }
                const int ir = iu + 8 * (v / 4) + (v % 4);  // uniform; the lane's row is ir + 4*half
                if (CHECK && not_ours(ir)) continue;
#pragma unroll
                for (int b = 0; b < TN; ++b) {
                    if (CHECK && !own[b]) continue;
                    float *c = reinterpret_cast<float *>(out + (long)ir * row_bytes + voff[b]);
                    float val = acc[a][b][v] * alpha + (MODE != 0 ? bias_v[v] + col_bias[b] : 0.0f);
                    if constexpr (MODE == 2) val += g.beta * held[v % ROWS][b];
                    if (act) val = val > g.act_threshold ? val : g.act_value;
                    if (masked) {
                        const float mv = *reinterpret_cast<const float *>(msk + (long)ir * mask_row_bytes + mvoff[b]);
                        val = mv > g.mask_threshold ? val : 0.0f;
                    }
                    *c = val;
                    if (twin) *reinterpret_cast<float *>(out2 + (long)ir * twin_row_bytes + tvoff[b]) = val;
                }
            }
        }
    };
    // The scattered store (see GemmProblem::scatter): rows are (plane, row phase, column phase) triples, columns
    // cells of a per-image grid; an element lands at a strided position of the image or is dropped.
    auto write_scatter = [&]() {
        const bool masked = g.mask != nullptr;
        long cbase[TN];  // float offset of the cell's phase-(0,0) pixel; may lie before the image (pH, pW)
        int hy[TN], wx[TN];
        bool own[TN];
#pragma unroll
        for (int b = 0; b < TN; ++b) {
            const int jt = j0 + wn * (TN * 32) + b * 32 + l32;
            own[b] = jt >= own_j0 && (!SHORT_J || jt < g.J);
            const int jg = col_at(jt);
            unsigned im, n, y, x;
            g.divN.divmod((unsigned)jg, im, n);
            g.divCW.divmod(n, y, x);
            hy[b] = (int)y * g.scat_sH - g.scat_pH;
            wx[b] = (int)x * g.scat_sW - g.scat_pW;
            cbase[b] = (long)im * g.bsC + (long)hy[b] * g.scat_W + wx[b];
        }
        const long plane = (long)g.scat_H * g.scat_W;
#pragma unroll
        for (int a = 0; a < TM; ++a) {
            const int iu = i0 + wm * (TM * 32) + a * 32;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = iu + 8 * (v / 4) + (v % 4) + 4 * half;
                if (row < own_i0 || row >= g.scat_rows) continue;
                unsigned c, rem, ph, pw;
                g.divScatS.divmod((unsigned)row, c, rem);
                g.divScatW.divmod(rem, ph, pw);
                const long roff = (long)c * plane + (long)ph * g.scat_W + pw;
#pragma unroll
                for (int b = 0; b < TN; ++b) {
                    const int h = hy[b] + (int)ph, w = wx[b] + (int)pw;
                    if (!own[b] || h < 0 || h >= g.scat_H || w < 0 || w >= g.scat_W) continue;
                    const long off = cbase[b] + roff;
                    float val = acc[a][b][v] * (column_sign * g.alpha) + 0.0f;
                    if (masked) val = g.mask[off] > g.mask_threshold ? val : 0.0f;
                    g.C[off] = val;
                }
            }
        }
    };
    if constexpr (RED) {
        if (rs_on) {
            const long slots = (long)g.nsplit * g.tilesJ;
            float *dst = g.rowsum_ws + ((long)split * g.tilesJ + tj);
#pragma unroll
            for (int q = 0; q < RS; ++q) {
                float total = bsum[q] + __shfl_xor(bsum[q], 1);  // four lanes hold the quarters of a row
                total += __shfl_xor(total, 2);
                const int row = i0 + a_x + q * (NT / 4);
                if (a_r == 0 && a_x + q * (NT / 4) < BM && row >= own_i0 && (!SHORT_M || row < g.M)) dst[row * slots] = total;
            }
        }
    }
    using std::integral_constant;
    if constexpr (LB == LD_XC_GATHER && !RED) {
        if (g.scatter) {
            write_scatter();
            return;
        }
    }
    if (g.nsplit > 1) {
        if (edge_tile) write_out(integral_constant<int, 0>{}, integral_constant<bool, true>{});
        else write_out(integral_constant<int, 0>{}, integral_constant<bool, false>{});
    } else if (g.beta == 0.0f) {
        if (edge_tile) write_out(integral_constant<int, 1>{}, integral_constant<bool, true>{});
        else write_out(integral_constant<int, 1>{}, integral_constant<bool, false>{});
    } else {
        if (edge_tile) write_out(integral_constant<int, 2>{}, integral_constant<bool, true>{});
        else write_out(integral_constant<int, 2>{}, integral_constant<bool, false>{});
    }
}

template <int BM, int BN, int WGM, int WGN, int LA, int LB, bool RED, int KG, bool FOLD = false>
__global__ __launch_bounds__(WGM *WGN * 64 * KG)
    __attribute__((amdgpu_waves_per_eu(KG > 1 ? KG : gemm_min_waves<BM, BN, WGM, WGN>()))) void gemm_fast_kernel(const GemmArgs g) {
    __shared__ __attribute__((aligned(16))) char As[KG * 2 * PartTile<BM>::kBytes];
    __shared__ __attribute__((aligned(16))) char Bs[KG * 2 * PartTile<BN>::kBytes];
    gemm_fast_tile<BM, BN, WGM, WGN, LA, LB, RED, KG, FOLD>(g, blockIdx.x, As, Bs);
}

// The workgroups of two products on the 64 x 64 tile of four groups, one after the other's.
template <int LA, int LB, bool RED, int LA2, int LB2, bool RED2>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(4))) void gemm_pair_kernel(const GemmArgs a, const GemmArgs b) {
    __shared__ __attribute__((aligned(16))) char As[4 * 2 * PartTile<64>::kBytes];
    __shared__ __attribute__((aligned(16))) char Bs[4 * 2 * PartTile<64>::kBytes];
    if (blockIdx.x < a.total) gemm_fast_tile<64, 64, 2, 2, LA, LB, RED, 4>(a, blockIdx.x, As, Bs);
    else gemm_fast_tile<64, 64, 2, 2, LA2, LB2, RED2, 4>(b, blockIdx.x - a.total, As, Bs);
}

template <int BM, int BN, int WGM, int WGN, int LA, int LB, bool RED, int KG = 1, bool FOLD = false>
int gemm_fast_go(const GemmArgs &g, hipStream_t s) {
    hipLaunchKernelGGL((gemm_fast_kernel<BM, BN, WGM, WGN, LA, LB, RED, KG, FOLD>), dim3(g.total), dim3(WGM * WGN * 64 * KG), 0, s, g);
    return 0;
}

// Dispatch over the loader kinds for one tile configuration.
template <int BM, int BN, int WGM, int WGN, int KG = 1>
int gemm_fast_dispatch(const GemmArgs &g, int la, int lb, bool red, hipStream_t s) {
#define THGPU_CASE(LA_, LB_)                                                           \
    if (la == LA_ && lb == LB_) {                                                      \
        if constexpr ((LA_ == LD_XC_SCALAR && (WGM * WGN * 64) % BM != 0 &&            \
                       !((WGM * WGN * 64) == 256 && BM % 64 == 0)) ||                  \
                      ((LB_ == LD_XC_SCALAR || LB_ == LD_XC_GATHER) && (WGM * WGN * 64) % BN != 0)) { \
            return fail("gemm: this tile has no x-contiguous loader for that side");   \
        } else {                                                                       \
            if (red) {                                                                 \
                if constexpr (LA_ == LD_RC_VEC && LB_ != LD_XC_SCALAR && LB_ != LD_XC_GATHER) \
                    return gemm_fast_go<BM, BN, WGM, WGN, LA_, LB_, true, KG>(g, s);     \
                else                                                                   \
                    return fail("gemm: reduction batching needs operands loaded along r"); \
            }                                                                          \
            if constexpr (LB_ == LD_RC_GATHER || LB_ == LD_RC_GATHER_VEC)              \
                return fail("gemm: a gather along r needs reduction batching");        \
            else                                                                       \
                return gemm_fast_go<BM, BN, WGM, WGN, LA_, LB_, false, KG>(g, s);        \
        }                                                                              \
    }
    THGPU_CASE(LD_RC_VEC, LD_RC_VEC)
    THGPU_CASE(LD_RC_VEC, LD_XC_SCALAR)
    THGPU_CASE(LD_RC_VEC, LD_XC_GATHER)
    THGPU_CASE(LD_RC_VEC, LD_RC_GATHER)
    THGPU_CASE(LD_RC_VEC, LD_RC_GATHER_VEC)
    THGPU_CASE(LD_XC_SCALAR, LD_RC_VEC)
    THGPU_CASE(LD_XC_SCALAR, LD_XC_SCALAR)
#undef THGPU_CASE
    return fail("gemm: unknown loader combination (%d, %d)", la, lb);
}

}  // namespace thgpu
