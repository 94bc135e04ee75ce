// Host side of the fp32 GEMM: picks a tile configuration, the operand
// loaders and a reduction split for a GemmProblem, launches the kernel and,
// when the reduction was split, the fixed-order reduction of the partial sums.
// Also the THGPUBlas_gemm entry point.
#include "gemm_mfma.h"
#include "side_jobs.h"

#include <cstring>
#include <map>
#include <mutex>
#include <new>

namespace thgpu {

namespace {

// C(i, j) = beta*C + alpha * sum_s ws[s][i][j] (+ bias[i]), s ascending; j is
// mapped through (image, n) when the output is column batched.
// The second job of a reduction launch: out[i] += alpha * sum over slots of ws[i][slot].  One wavefront per row:
// lane l adds slots l, l + 64, ... in ascending order, then the lanes are added pairwise in a fixed tree, so the
// result is reproducible.
struct RowSumJob {
    const float *ws;
    float *out;
    int M, slots;
    float alpha;
};

__device__ __forceinline__ void rowsum_reduce(const RowSumJob &j, unsigned block) {
    const int lane = threadIdx.x & 63;
    const int row = (int)block * 4 + (int)(threadIdx.x >> 6);
    if (row >= j.M) return;  // a whole wavefront
    const float *src = j.ws + (long)row * j.slots;
    float sum = 0.0f;
    for (int s = lane; s < j.slots; s += 64) sum += src[s];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) sum += __shfl_down(sum, d);
    if (lane == 0) j.out[row] += j.alpha * sum;
}

// The reduction of one product's partial sums and whatever rides with it.
//
// In the order in which a wavefront needs it: it lives for 2 us, of which a second round of scalar loads before the partial
// sums can be asked for is a tenth (14 reductions of a VGG-A step: 607 us, 643 with the row sums' job in front).
struct ReduceJob {
    unsigned rowsum_first_block, side_first_block;  // workgroups from these on do the jobs at the end
    unsigned total;                                 // outputs: M*J
    int nsplit;
    const float *ws;
    float *C;
    FastDiv divJ;
    unsigned j_store;
    int J, N;
    long sC, bsC;
    const float *bias, *bias_col, *mask;
    float *C2;
    float alpha, beta;
    int act;
    float act_threshold, act_value, mask_threshold;
    int c_pitch, mask_pitch, c2_pitch;
    FastDiv divN, divCW;
    long mask_sC, mask_bsC, c2_sC, c2_bsC;
    unsigned blocks;
    bool quarters;
    RowSumJob rs;
    WeightJob side;  // a job of the next layer's (side_jobs.h)
};

template <bool quarters>
__device__ __forceinline__ void split_reduce(const ReduceJob &j, unsigned block) {
    if (block >= j.side_first_block) {
        reorder_weight(j.side, (block - j.side_first_block) * 256u + threadIdx.x);
        return;
    }
    if (block >= j.rowsum_first_block) {
        rowsum_reduce(j.rs, block - j.rowsum_first_block);
        return;
    }
    // With `quarters` the four wavefronts of a workgroup share 64 outputs, each adding a contiguous quarter of the
    // partial sums (for few outputs and many splits: one lane per output would leave the GPU idle behind a long
    // chain of loads); the quarters are then added in order.  Either way the order of the adds is fixed.
    const unsigned total = j.total;
    const unsigned wave = threadIdx.x >> 6;
    unsigned idx = quarters ? block * 64u + (threadIdx.x & 63u) : block * 256u + threadIdx.x;
    const bool valid = idx < total;
    if (!quarters && !valid) return;
    const int per = quarters ? (j.nsplit + 3) / 4 : j.nsplit;
    const int s_begin = quarters ? (int)wave * per : 0;
    const int s_end = s_begin + per < j.nsplit ? s_begin + per : j.nsplit;
    // Eight partials are requested before the first is added; the adds stay in split order.
    float sum = 0.0f;
    const float *src = j.ws + (valid ? idx : 0);
    for (int s0 = s_begin; s0 < s_end; s0 += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = s0 + u < s_end ? src[(long)(s0 + u) * total] : 0.0f;
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (s0 + u < s_end) sum += v[u];
    }
    if (quarters) {
        __shared__ float part[4][64];
        part[wave][threadIdx.x & 63u] = sum;
        __syncthreads();
        if (wave != 0 || !valid) return;
        sum = ((part[0][threadIdx.x] + part[1][threadIdx.x]) + part[2][threadIdx.x]) + part[3][threadIdx.x];
    }
    unsigned row, col;
    j.divJ.divmod(idx, row, col);
    if (col >= j.j_store) return;  // a scratch column of a product run wider than its result (GemmProblem::j_store)
    long coff = col, moff = col, toff = 0;
    if (j.N != j.J || j.c_pitch || j.mask_pitch || j.C2) {
        unsigned im, n, y, x;
        j.divN.divmod(col, im, n);
        j.divCW.divmod(n, y, x);
        coff = (long)im * j.bsC + (j.c_pitch ? (long)y * j.c_pitch + x : (long)n);
        moff = (long)im * j.mask_bsC + (j.mask_pitch ? (long)y * j.mask_pitch + x : (long)n);
        toff = (long)im * j.c2_bsC + (long)y * j.c2_pitch + x;
    }
    float *c = j.C + (long)row * j.sC + coff;
    float val = j.alpha * sum;
    if (j.bias) val += j.bias[row];
    if (j.bias_col) val += j.bias_col[col];
    if (j.beta != 0.0f) val += j.beta * *c;
    if (j.act) val = val > j.act_threshold ? val : j.act_value;
    if (j.mask) val = j.mask[(long)row * j.mask_sC + moff] > j.mask_threshold ? val : 0.0f;
    *c = val;
    if (j.C2) j.C2[(long)row * j.c2_sC + toff] = val;  // the second copy (GemmProblem::C2)
}

template <bool quarters>
__global__ __launch_bounds__(256) void split_reduce_kernel(const ReduceJob j) {
    split_reduce<quarters>(j, blockIdx.x);
}

// Two products' reductions in one launch.
__global__ __launch_bounds__(256) void split_reduce_pair_kernel(const ReduceJob a, const ReduceJob b) {
    if (blockIdx.x < a.blocks) {
        if (a.quarters) split_reduce<true>(a, blockIdx.x);
        else split_reduce<false>(a, blockIdx.x);
    } else {
        if (b.quarters) split_reduce<true>(b, blockIdx.x - a.blocks);
        else split_reduce<false>(b, blockIdx.x - a.blocks);
    }
}

struct TileCfg {
    const char *name;
    int bm, bn;
    int resident;  // workgroups that fit a CU at once (registers / LDS)
    // Fraction of the MFMA rate (kFlopsPerCycle) the inner loop sustains with a full CU, by operand layout: [0] A along r,
    // B along j (forward); [1] both along their free index (gradInput); [2] both along r (gradWeight); [3] A along i, B
    // along r; [4] A along r, B gathered; [5] the same with reduction batching.
    // Measured like the occupancy tables below.  None is near 1: on uniform random operands these kernels are held by the
    // card's power, not by its issue slots (the clock falls to about 1.6 GHz; the same launches on zeros run a fifth
    // faster), as is the library's bf16 product (1.13 PFLOP/s at 8192^3, which is 189 TFLOP/s at six products each).
    double eff[6];
    int (*launch)(const GemmArgs &, int, int, bool, hipStream_t);
    // Fraction of that rate kept with k = 1..4 workgroups resident per CU, and the row count from which the tile is no
    // longer considered (0: no limit).
    const double *occ;
    int below_rows;
    // The tile has no loader for a first operand contiguous along its rows.
    bool a_rc_only;
    // Groups of wavefronts that share a workgroup's reduction (gemm_fast.h, finish_groups).
    int groups = 1;
    bool folds = false;  // sums in two levels (gemm_fold_steps)
};

// Rate kept with k workgroups on a CU, by tile: measured on 3x3 forward products of 2304 reduction indices and exactly
// k workgroups per CU (128 x 128: 102, 152, 165 TFLOP/s with one, two, three).
const double kOcc2[5] = {0.0, 0.77, 1.0};
const double kOcc3[5] = {0.0, 0.60, 0.91, 1.0};
const double kOcc4[5] = {0.0, 0.57, 0.81, 0.95, 1.0};
const double kOccSmall[5] = {0.0, 0.43, 0.75, 0.91, 1.0};
const double kOcc1[2] = {0.0, 1.0};

const TileCfg kCfgs[] = {
    {"128x128", 128, 128, 3, {0.38, 0.38, 0.38, 0.38, 0.39, 0.38}, gemm_fast_128x128, kOcc3, 0, false},
    {"192x128", 192, 128, 2, {0.41, 0.41, 0.41, 0.41, 0.42, 0.40}, gemm_fast_192x128, kOcc2, 0, false},
    {"64x256", 64, 256, 2, {0.31, 0.31, 0.31, 0.31, 0.32, 0.30}, gemm_fast_64x256, kOcc2, 0, false},
    {"128x256", 128, 256, 2, {0.39, 0.39, 0.39, 0.39, 0.40, 0.38}, gemm_fast_128x256, kOcc2, 0, false},
    {"256x128", 256, 128, 2, {0.42, 0.42, 0.42, 0.42, 0.43, 0.44}, gemm_fast_256x128, kOcc2, 0, false},
    {"64x64", 64, 64, 4, {0.29, 0.29, 0.29, 0.29, 0.30, 0.25}, gemm_fast_64x64, kOccSmall, 0, false},
    {"64x128", 64, 128, 4, {0.33, 0.33, 0.33, 0.33, 0.34, 0.33}, gemm_fast_64x128, kOcc4, 128, false},
    {"96x128", 96, 128, 3, {0.35, 0, 0.35, 0, 0.37, 0.35}, gemm_fast_96x128, kOcc3, 128, true},
    {"32x128", 32, 128, 4, {0.22, 0, 0.22, 0, 0.22, 0.25}, gemm_fast_32x128, kOcc4, 33, true},
    {"64x64f", 64, 64, 4, {0, 0, 0, 0, 0.29, 0}, gemm_fast_64x64f, kOccSmall, 0, true, 1, true},
    {"64x64k4", 64, 64, 1, {0.25, 0.25, 0.25, 0.25, 0.26, 0.27}, gemm_fast_64x64k4, kOcc1, 0, false, 4},
};

inline long cdiv(long a, long b) { return (a + b - 1) / b; }

// Flops a CU retires per cycle with six bf16 products for one fp32 product: 4096 / 6.
constexpr double kFlopsPerCycle = 4096.0 / 6.0;

// Rough time model (in CU-cycles) used only to rank (tile, split) candidates.
// A CU retires kFlopsPerCycle flops at best; with fewer workgroups resident it
// hides less of their latencies (kOcc); workgroups beyond what fits at once
// run in further rounds; every round pays a prologue/epilogue; a split adds
// the traffic of writing and re-reading the partial sums.
double model_cycles(const TileCfg &c, int layout, long M, long J, long steps_total, int nsplit, int cus, bool accumulate) {
    const double *kOcc = c.occ;
    const long tiles = cdiv(M, c.bm) * cdiv(J, c.bn);
    const long wgs = tiles * nsplit;
    const long steps = cdiv(cdiv(steps_total, nsplit), c.groups) * c.groups;
    const double per_step = 2.0 * c.bm * c.bn * GEMM_BK / kFlopsPerCycle / c.eff[layout];
    const long slots = (long)cus * c.resident;
    const long full = wgs / slots, rest = wgs - full * slots;
    // (A workgroup of groups has its CU to itself: where more than one follows another, nothing runs under its first loads and
    // its stores: 395 x 3740 over 648, 413 tiles: 45.4 us, 37.3 with 64 x 64 tiles.)
    const double ovh = 3000.0 + 6.0 * c.bm * c.bn / 64.0 + (c.groups > 1 && wgs > slots ? 6000.0 : 0.0);
    // A CU stores an output in half a cycle (4.8 TB/s over the chip); where a reduction is too short to hide that, a round
    // takes what its tiles' stores take and, at its start, one tile's more (20 indices, 225 x 161772: 64 us with two 128 x 256
    // tiles to a CU, 42 us with four of 64 x 128; an accumulating store also reads).
    const double stores = 0.55 * c.bm * c.bn * (accumulate ? 2.0 : 1.0);
    auto at_least = [](double a, double b) { return a > b ? a : b; };
    const double round = at_least(c.resident * steps * per_step / kOcc[c.resident] + ovh, (c.resident + 1) * stores);
    double t = full * round;
    if (rest > 0) {
        const long on_busiest = cdiv(rest, cus);
        const int k = (int)(on_busiest < c.resident ? on_busiest : c.resident);
        double last = at_least(on_busiest * steps * per_step / kOcc[k] + ovh * (k > 1 ? 1.0 : 1.5), (on_busiest + 1) * stores);
        // Behind full rounds a thin last one costs half of what it would alone: workgroups do not end in step, and the
        // last ones run at the clock that an idle chip allows (512 x 50176 over 2304, 128 x 128 tiles: 2.04 rounds,
        // 816 us with the last counted in full, measured 620; in three parts, 2.3 rounds of larger tiles, 561 us and
        // 114 for the partial sums).
        if (full > 0) last = 0.5 * (last + round * rest / slots);
        t += last;
    }
    if (c.groups > 1) t += 1000.0;  // the groups' sums through LDS
    if (nsplit > 1) t += 5000.0 + (double)(nsplit + 2) * M * J * 4.0 / (4.5e12 / 2.4e9);  // launch, bytes / (bytes per cycle)
    return t;
}

// Few outputs and many splits: four wavefronts share 64 outputs of the split reduction (reduce_job).
inline bool reduced_in_quarters(long outputs, int nsplit) { return outputs > 0 && outputs < 128 * 1024 && nsplit >= 12; }

// What one output of a plan is rounded, level by level (gemm_roundings): a wavefront's steps, its workgroup's groups, the parts.
double plan_roundings(const TileCfg &c, long outputs, int steps_total, int nsplit) {
    const long part = cdiv(steps_total, nsplit), walk = cdiv(part, c.groups);
    const int f = gemm_fold_steps((int)walk);
    double n = c.folds && f < walk ? gemm_roundings(f) + gemm_roundings((double)walk / f) : gemm_roundings((double)walk);
    if (c.groups > 1 && walk > 0) n += gemm_roundings((double)cdiv(part, walk));
    if (nsplit > 1)
        n += reduced_in_quarters(outputs, nsplit) ? gemm_roundings((double)cdiv(nsplit, 4)) + gemm_roundings(4) : gemm_roundings(nsplit);
    return n;
}

// The tile configuration and reduction split for a problem; cfg == nullptr when no tiled kernel takes it.
struct GemmPlan {
    const TileCfg *cfg = nullptr;
    int nsplit = 1;
    double cycles = 0;  // the model's estimate
};

// `any`: the first tile and split that can run the problem, without ranking them.
GemmPlan rank_plans(const GemmProblem &p, int steps_total, bool any) {
    GemmPlan plan;
    const bool gather = p.rowtab != nullptr;
    const int cus = num_cus();
    double best_t = 0;
    // Tuning aids: the gemm_tile switch forces a configuration by name, gemm_split a split count.
    const Tuning &tune = tuning();
    const char *force = tune.gemm_tile[0] ? tune.gemm_tile : nullptr;
    const int fsplit = tune.gemm_split;
    // The fast kernel addresses each operand as a uniform base plus a 32-bit
    // per-thread byte offset and moves a partial last step back by up to 15
    // reduction indices: it needs R >= 16 and tile-local offsets below 2^30 floats.
    // The output is addressed the same way (four rows and a tile's columns per lane).
    const long n_img = p.N > 0 ? p.N : p.J;
    auto offsets_fit = [&](int bm, int bn) {
        const long offA = p.a_rc ? (long)(bm - 1) * p.sA + GEMM_BK : (long)(GEMM_BK - 1) * p.sA + bm;
        const long span = (bn - 1) / n_img + 2;  // images a tile's columns can touch
        const long offB = gather ? p.b_extent
                          : p.b_rc ? (long)(bn - 1) * p.sB + GEMM_BK
                                   : (long)(GEMM_BK - 1) * p.sB + span * p.bsB + n_img;
        const long offC = 4 * (p.sC > p.J ? p.sC : (long)p.J) + span * p.bsC + n_img;
        const long offC2 = p.C2 ? 4 * p.c2_sC + span * p.c2_bsC + (p.c_w > 0 ? n_img / p.c_w : 0) * p.c2_pitch + p.c_w : 0;
        return offA < (1L << 30) && offB < (1L << 30) && offC < (1L << 30) && offC2 < (1L << 30);
    };
    const bool fast_ok = p.R == 0 || p.R >= GEMM_BK;
    const int layout = gather ? (p.nb > 1 || p.rowsum ? 5 : 4) : p.a_rc ? (p.b_rc ? 2 : 0) : (p.b_rc ? 3 : 1);
    for (const TileCfg &c : kCfgs) {
        if (!fast_ok || !offsets_fit(c.bm, c.bn)) continue;
        if ((p.M < c.bm && c.bm > GEMM_SHORT_TILE) || (p.J < c.bn && c.bn > GEMM_SHORT_TILE)) continue;
        if (force && std::strcmp(force, c.name) != 0) continue;
        if (!force && c.below_rows > 0 && p.M >= c.below_rows) continue;
        if (c.a_rc_only && !p.a_rc) continue;
        if (c.folds && (layout != 4 || (!force && p.max_roundings < 0.0))) continue;
        const double best_roundings = plan.cfg ? plan_roundings(*plan.cfg, (long)p.M * p.J, steps_total, plan.nsplit) : 0.0;
        const long tiles = cdiv(p.M, c.bm) * cdiv(p.J, c.bn);
        // (a product run wider than its result has one narrow tile per row block: it may split further to fill the GPU)
        const int split_cap = p.j_store > 0 ? 1024 : 256;
        int max_split = (int)(steps_total / 8 > 0 ? (steps_total / 8 < split_cap ? steps_total / 8 : split_cap) : 1);
        if (p.scatter) max_split = 1;  // the scattered store has no partial-sum form
        const int min_split = p.j_store > 0 ? 2 : 1;  // scratch columns never reach C unsplit
        int want = fsplit > 0 ? (fsplit < max_split ? fsplit : max_split) : 0;
        if (want > 0 && want < min_split) want = min_split;
        for (int ns = min_split; ns <= max_split; ++ns) {
            if (want > 0 && ns != want) continue;
            if (tiles * ns > 8L * cus * c.resident && ns > 1 && fsplit <= 0) break;
            if (ns > 1 && p.ws_fixed && (long)ns * p.M * p.J > p.ws_fixed_floats) break;  // partial sums must fit
            const int sps = (int)cdiv(steps_total, ns);
            if (sps > 0 && (int)cdiv(steps_total, sps) != ns) continue;  // would leave an empty split
            if (!force && fsplit <= 0) {
                const double roundings = plan_roundings(c, (long)p.M * p.J, steps_total, ns);
                if (p.max_roundings >= 0.0 && roundings > p.max_roundings) continue;
                // (the tile of groups, the last one, does with fewer parts what the others split further: not at the price of
                // longer sums, 282 x 294 over 2272 steps in 85 parts 1.41e-7 from 64 bits, in 10 of four groups 1.61e-7)
                if (c.groups > 1 && plan.cfg && roundings > best_roundings) continue;
            }
            if (any) {
                plan.cfg = &c;
                plan.nsplit = ns;
                return plan;
            }
            const double t = model_cycles(c, layout, p.M, p.J, steps_total, ns, cus, p.beta != 0.0f);
            if (!plan.cfg || t < best_t) {
                best_t = t;
                plan.cfg = &c;
                plan.nsplit = ns;
                plan.cycles = t;
            }
        }
    }
    return plan;
}

// What the planner's answer depends on.
struct PlanKey {
    long v[22];
    bool operator<(const PlanKey &o) const { return std::memcmp(v, o.v, sizeof(v)) < 0; }
};

// Ranking walks up to a thousand splits of eight tiles, 3 to 20 us, more than a launch takes to enqueue, and a program asks
// for the same few products in every pass: the answers are kept by shape (host time of an AlexNet-style step, together with
// gemm_tiled_fits, which no longer ranks: 285 -> 189 us; first-layer shape, three passes: 43 -> 30 us).  At 4096 shapes the map
// starts over.
GemmPlan plan_gemm(const GemmProblem &p, int steps_total) {
    const Tuning &tune = tuning();
    if (tune.gemm_tile[0] || tune.gemm_split > 0) return rank_plans(p, steps_total, false);
    static std::mutex mutex;
    static std::map<PlanKey, GemmPlan> plans;
    const PlanKey key = {{p.M, p.J, p.R, p.N, steps_total, p.nb > 1 || p.rowsum,
                          (p.a_rc ? 1 : 0) + (p.b_rc ? 2 : 0) + (p.rowtab ? 4 : 0) + (p.scatter ? 8 : 0) + (p.C2 ? 16 : 0), p.j_store,
                          p.sA, p.sB, p.sC, p.bsB, p.bsC, p.b_extent, p.C2 ? p.c2_sC : 0, p.C2 ? p.c2_bsC : 0,
                          p.C2 ? p.c2_pitch : 0, p.C2 ? p.c_w : 0, p.ws_fixed ? 1 : 0, p.ws_fixed ? p.ws_fixed_floats : 0, p.beta != 0.0f,
                          (long)(4096.0 * p.max_roundings)}};
    {
        std::lock_guard<std::mutex> lock(mutex);
        const auto it = plans.find(key);
        if (it != plans.end()) return it->second;
    }
    const GemmPlan plan = rank_plans(p, steps_total, false);
    try {
        std::lock_guard<std::mutex> lock(mutex);
        if (plans.size() >= 4096) plans.clear();
        plans[key] = plan;
    } catch (const std::bad_alloc &) {  // not kept, then
    }
    return plan;
}

inline int steps_of(const GemmProblem &p) {
    return (p.R + GEMM_BK - 1) / GEMM_BK * (p.nb > 1 ? p.nb : 1);
}

}  // namespace

bool gemm_tiled_fits(const GemmProblem &p) {
    if (p.M <= 0 || p.J <= 0 || (long)p.M * p.J >= (1L << 31)) return false;
    // (where the first tile and split will not do, the answer is the planner's, which keeps it)
    return (p.max_roundings >= 0.0 ? plan_gemm(p, steps_of(p)) : rank_plans(p, steps_of(p), true)).cfg != nullptr;
}

double gemm_plan_roundings(const GemmProblem &p) {
    const GemmPlan plan = plan_gemm(p, steps_of(p));
    // (the generic kernel takes reductions of less than a step, which count as one term)
    return plan.cfg ? plan_roundings(*plan.cfg, (long)p.M * p.J, steps_of(p), plan.nsplit) : gemm_roundings(steps_of(p));
}

double gemm_estimate_us(const GemmProblem &p) {
    const GemmPlan plan = plan_gemm(p, steps_of(p));
    if (plan.cfg) return plan.cycles / 2400.0;
    // the generic kernel: 25 TFLOP/s over whole 64 x 64 tiles, or its stores
    const double compute = 2.0 * 64 * 64 * cdiv(p.M, 64) * cdiv(p.J, 64) * (double)p.R / 25e6;
    const double store = 4.0 * p.M * (double)p.J / 4.5e6;
    return 4.0 + (compute > store ? compute : store);
}

namespace {

// A product on its way: what its launches need besides the workspace.
struct Prepared {
    const GemmProblem *p;
    GemmArgs g;
    const TileCfg *best;  // nullptr: the generic kernel
    int la, lb;
    bool red, rowsum;
    size_t ws_floats, rowsum_floats;  // of partial sums and partial row sums together, of the latter
};

int gemm_prepare(const GemmProblem &p, Prepared &out) {
    if ((long)p.M * p.J >= (1L << 31)) return fail("gemm: output of %d x %d exceeds 32-bit tile indexing", p.M, p.J);

    // (one image's gradWeight runs as a reduction batch of one where it wants the row sums of A)
    const bool red = p.nb > 1 || (p.rowsum && p.a_rc && (p.b_rc || p.rowtab));
    const bool gather = p.rowtab != nullptr;
    if (gather && (!p.coltab || p.b_rc || !p.a_rc)) return fail("gemm: a gathered B needs both tables and an r-contiguous A");
    if (red && !(p.a_rc && (p.b_rc || gather))) return fail("gemm: reduction batching needs r-contiguous operands");

    GemmArgs &g = out.g;
    std::memset(&g, 0, sizeof(g));
    g.A = p.A;
    g.B = p.B;
    g.C = p.C;
    g.bias = p.bias;
    g.bias_col = p.bias_col;
    if (p.bias_col && (p.bias || red || gather || p.C2 || (p.N > 0 && p.N != p.J)))
        return fail("gemm: a bias per column needs a plain product");
    g.rowtab = p.rowtab;
    g.coltab = p.coltab;
    g.M = p.M;
    g.J = p.J;
    g.R = p.R;
    g.N = p.N > 0 ? p.N : p.J;
    g.sA = p.sA;
    g.sB = p.sB;
    g.sC = p.sC;
    g.bsB = p.bsB;
    g.bsC = p.bsC;
    g.rbA = p.rbA;
    g.rbB = p.rbB;
    g.nb = p.nb;
    g.divN = FastDiv((uint32_t)g.N);
    g.alpha = p.alpha;
    g.beta = p.beta;
    g.act = p.act ? 1 : 0;
    g.act_threshold = p.act_threshold;
    g.act_value = p.act_value;
    g.mask = p.mask;
    g.mask_threshold = p.mask_threshold;
    if ((p.c_pitch || p.mask_pitch) && (p.c_w <= 0 || red || g.N % p.c_w != 0))
        return fail("gemm: pitched rows need column batching and a plane width that divides the columns of an image");
    g.c_w = p.c_w > 0 ? p.c_w : 1;
    g.c_pitch = p.c_pitch;
    g.mask_pitch = p.mask_pitch;
    g.mask_sC = p.mask_sC ? p.mask_sC : p.sC;
    g.mask_bsC = p.mask_bsC ? p.mask_bsC : p.bsC;
    g.divCW = FastDiv((uint32_t)g.c_w);
    // (reduction batching or one image: either way every column of the product is a column of C or scratch)
    if (p.j_store > 0 && (p.N != p.J || p.j_store > p.J || p.sC < p.j_store || p.C2 || p.scatter))
        return fail("gemm: scratch columns need an unbatched column index and a row pitch of C that holds the stored ones");
    if (p.C2) {
        if (red || p.scatter || p.c_w <= 0 || g.N % p.c_w != 0 || p.c2_pitch < p.c_w || p.c2_sC <= 0 || p.c2_bsC <= 0)
            return fail("gemm: a second copy of the result needs column batching, a plane width and the copy's strides");
        g.C2 = p.C2;
        g.c2_sC = p.c2_sC;
        g.c2_bsC = p.c2_bsC;
        g.c2_pitch = p.c2_pitch;
    }
    if (p.scatter) {
        if (!gather || red || p.bias || p.beta != 0.0f || p.c_pitch || p.mask_pitch || p.c_w <= 0 || g.N % p.c_w != 0 ||
            p.scat_sH <= 0 || p.scat_sW <= 0 || p.scat_H <= 0 || p.scat_W <= 0 || p.scat_rows <= 0 || p.scat_rows > p.M ||
            p.scat_pH < 0 || p.scat_pW < 0)
            return fail("gemm: a scattered store needs a gathered B, column batching, no bias and beta = 0");
        g.scatter = 1;
        g.scat_sH = p.scat_sH;
        g.scat_sW = p.scat_sW;
        g.scat_pH = p.scat_pH;
        g.scat_pW = p.scat_pW;
        g.scat_H = p.scat_H;
        g.scat_W = p.scat_W;
        g.scat_rows = p.scat_rows;
        g.divScatS = FastDiv((uint32_t)(p.scat_sH * p.scat_sW));
        g.divScatW = FastDiv((uint32_t)p.scat_sW);
    }
    g.steps_per_img = (p.R + GEMM_BK - 1) / GEMM_BK;
    g.steps_total = g.steps_per_img * (red ? p.nb : 1);
    g.divSpi = FastDiv((uint32_t)(g.steps_per_img > 0 ? g.steps_per_img : 1));

    const int cus = num_cus();
    const GemmPlan plan = plan_gemm(p, g.steps_total);
    const TileCfg *best = plan.cfg;
    const int best_split = plan.nsplit;

    g.nsplit = best ? best_split : 1;
    const int bm = best ? best->bm : 64, bn = best ? best->bn : 64;
    if (!best && !p.scatter && g.steps_total > 0) {
        // The generic kernel splits too: enough workgroups to fill the chip, eight steps each at least.  One workgroup per
        // 64 x 64 tile would walk the whole reduction of a small product alone (50 x 128 over 4096, a Linear layer
        // behind a small net: 144 us unsplit, 14 us in 32 parts).
        const long tiles = cdiv(p.M, 64) * cdiv(p.J, 64);
        long want = cdiv(2L * cus, tiles);
        const long cap = g.steps_total / 8 > 0 ? g.steps_total / 8 : 1;
        if (want > cap) want = cap;
        if (want < 1) want = 1;
        if (p.ws_fixed && want * p.M * p.J > p.ws_fixed_floats) want = p.ws_fixed_floats / ((long)p.M * p.J);
        if (want < 1) want = 1;
        const int sps = (int)cdiv(g.steps_total, want);
        g.nsplit = (int)cdiv(g.steps_total, sps);
    }
    g.steps_per_split = (int)cdiv(g.steps_total, g.nsplit);
    g.fold_steps = gemm_fold_steps(g.steps_per_split);
    g.tilesM = (unsigned)cdiv(p.M, bm);
    g.tilesJ = (unsigned)cdiv(p.J, bn);
    g.divTilesM = FastDiv(g.tilesM);
    g.divTilesJ = FastDiv(g.tilesJ);
    const long total = (long)g.tilesM * g.tilesJ * g.nsplit;
    if (total <= 0 || total >= (1L << 31)) return fail("gemm: tile count %ld out of range", total);
    g.total = (unsigned)total;
    // Row sums of A ride along with a tiled reduction-batched product (never with the fixed workspace of the
    // entry point that may not allocate: nothing there asks for them).
    // (An unsplit product of few rows leaves them to their own launch, which reads as little and needs no scratch.)
    const bool rowsum = p.rowsum && best && red && !p.ws_fixed && (g.nsplit > 1 || p.M >= 64);
    if (p.rowsum_done) *p.rowsum_done = rowsum;
    out.rowsum_floats = rowsum ? (size_t)g.nsplit * g.tilesJ * p.M : 0;
    out.ws_floats = (g.nsplit > 1 ? (size_t)g.nsplit * p.M * p.J : 0) + out.rowsum_floats;
    if (p.ws_fixed && (long)out.ws_floats > p.ws_fixed_floats)
        return fail("gemm: %zu floats of partial sums exceed the fixed workspace of %ld", out.ws_floats, p.ws_fixed_floats);

    // ---- loaders: r-contiguous operands use 128-bit loads (4-byte alignment suffices) --------
    out.la = p.a_rc ? LD_RC_VEC : LD_XC_SCALAR;
    out.lb = p.b_rc ? LD_RC_VEC
                   : !gather ? LD_XC_SCALAR
                   : !red ? LD_XC_GATHER
                   : p.row_quads ? LD_RC_GATHER_VEC
                                 : LD_RC_GATHER;
    if (gather && !best) return fail("gemm: a gathered B needs a shape the tiled kernel takes (R >= 16)");
    if (p.C2 && !best) return fail("gemm: a second copy of the result needs a shape the tiled kernel takes");
    if (p.j_store > 0 && (!best || g.nsplit < 2))
        return fail("gemm: scratch columns need a tiled kernel and a split reduction");

    out.p = &p;
    out.best = best;
    out.red = red;
    out.rowsum = rowsum;
    return 0;
}

void use_workspace(Prepared &q, float *ws) {
    q.g.ws = ws;
    if (q.rowsum) q.g.rowsum_ws = ws + (q.ws_floats - q.rowsum_floats);
}

const char *product_label(const Prepared &q) {
    const GemmProblem &p = *q.p;
    return !prof_enabled() ? p.tag
                           : prof_label("%s M=%d J=%d R=%ld tile=%s split=%d", p.tag, p.M, p.J,
                                        (long)p.R * (q.red ? p.nb : 1), q.best ? q.best->name : "generic", q.g.nsplit);
}

double product_flops(const Prepared &q) {
    const GemmProblem &p = *q.p;
    return p.flops > 0 ? p.flops : 2.0 * p.M * p.J * (double)p.R * (q.red ? p.nb : 1);
}

int run_product(const Prepared &q, hipStream_t s) {
    const GemmProblem &p = *q.p;
    int rc;
    {
        LaunchScope scope(product_label(q), product_flops(q), 0.0);
        rc = q.best ? q.best->launch(q.g, q.la, q.lb, q.red, s) : gemm_generic_64x64(q.g, p.a_rc, p.b_rc, q.red, s);
    }
    return rc ? rc : check_launch(p.tag);
}

// The reduction behind a product that was split or sums rows on the side; returns its bytes for the timing.
double reduce_job(const Prepared &q, ReduceJob &job) {
    const GemmProblem &p = *q.p;
    const GemmArgs &g = q.g;
    std::memset(static_cast<void *>(&job), 0, sizeof(job));
    const long n = g.nsplit > 1 ? (long)p.M * p.J : 0;  // an unsplit product has stored its own result
    // few outputs, many splits: four wavefronts per 64 outputs.  From 4 K to 123 K outputs the launch alone takes the same
    // either way up to 16 splits, 0.2 us less at 24, 0.5 at 32 and 2.4 at 64; behind its product (256 x 169 outputs in 27
    // parts and two more like it, 3x3 layers of one 13x13 image) 12 as the line gave 53.1 -> 50.8 us a pass against 32.
    job.quarters = reduced_in_quarters(n, g.nsplit);
    job.blocks = (unsigned)cdiv(n, job.quarters ? 64 : 256);
    job.rowsum_first_block = job.blocks;  // four rows to a workgroup
    if (q.rowsum) {
        job.rs.ws = g.rowsum_ws;
        job.rs.out = p.rowsum;
        job.rs.M = p.M;
        job.rs.slots = (int)(g.nsplit * g.tilesJ);
        job.rs.alpha = p.alpha;
        job.blocks += (unsigned)cdiv(p.M, 4);
    }
    // A product that stores a second copy of its result for the next layer's gradInput product also carries that
    // layer's pending kernel-bank job, if there is one.
    job.side_first_block = job.blocks;
    double side_bytes = 0.0;
    if (g.C2 && n > 0 && take_bank_job(job.side)) {
        job.blocks += (job.side.count + 255u) / 256u;
        side_bytes = 4.0 * (job.side.count + (double)job.side.M * job.side.C * job.side.kH * job.side.kW);
    }
    job.ws = g.ws;
    job.C = p.C;
    job.bias = p.bias;
    job.bias_col = p.bias_col;
    job.total = (unsigned)p.M * (unsigned)p.J;
    job.J = p.J;
    job.N = g.N;
    job.sC = p.sC;
    job.bsC = p.bsC;
    job.divJ = FastDiv((uint32_t)p.J);
    job.divN = g.divN;
    job.divCW = g.divCW;
    job.nsplit = g.nsplit;
    job.alpha = p.alpha;
    job.beta = p.beta;
    job.act = g.act;
    job.act_threshold = g.act_threshold;
    job.act_value = g.act_value;
    job.mask = g.mask;
    job.mask_threshold = g.mask_threshold;
    job.c_pitch = g.c_pitch;
    job.mask_pitch = g.mask_pitch;
    job.mask_sC = g.mask_sC;
    job.mask_bsC = g.mask_bsC;
    job.C2 = g.C2;
    job.c2_sC = g.c2_sC;
    job.c2_bsC = g.c2_bsC;
    job.c2_pitch = g.c2_pitch;
    job.j_store = (unsigned)(p.j_store > 0 ? p.j_store : p.J);
    return 4.0 * n * (g.nsplit + 2 + (g.C2 ? 1 : 0)) + 4.0 * q.rowsum_floats + side_bytes;
}

int run_reduce(const ReduceJob &job, double bytes, hipStream_t s) {
    {
        LaunchScope scope("gemm_split_reduce", 0.0, bytes);
        auto kernel = job.quarters ? split_reduce_kernel<true> : split_reduce_kernel<false>;
        hipLaunchKernelGGL(kernel, dim3(job.blocks), dim3(256), 0, s, job);
    }
    return check_launch("gemm_split_reduce");
}

}  // namespace

int gemm_launch(const GemmProblem &p) {
    hipStream_t s = stream();
    if (!s) return 1;
    if (p.M <= 0 || p.J <= 0) return 0;
    Prepared q;
    if (gemm_prepare(p, q)) return 1;
    if (q.ws_floats > 0) {
        float *ws = p.ws_fixed ? p.ws_fixed : workspace(sizeof(float) * q.ws_floats);
        if (!ws) return 1;
        use_workspace(q, ws);
    }
    if (run_product(q, s)) return 1;
    if (q.ws_floats == 0) return 0;
    ReduceJob job;
    const double bytes = reduce_job(q, job);
    return run_reduce(job, bytes, s);
}

// Two products of which neither reads what the other writes.  Their split reductions share a launch, and where both are
// small enough for the tile of four groups, so do they themselves: a launch is 3 us to enqueue and 3 to 5 for the GPU to
// run and change over, as long as such a product takes.
int gemm_launch_pair(const GemmProblem &a, const GemmProblem &b) {
    hipStream_t s = stream();
    if (!s) return 1;
    if (a.M <= 0 || a.J <= 0 || b.M <= 0 || b.J <= 0 || a.ws_fixed || b.ws_fixed) return gemm_launch(a) || gemm_launch(b) ? 1 : 0;
    Prepared qa, qb;
    if (gemm_prepare(a, qa) || gemm_prepare(b, qb)) return 1;
    const size_t first = (qa.ws_floats + 63) / 64 * 64;
    if (first + qb.ws_floats > 0) {
        float *ws = workspace(sizeof(float) * (first + qb.ws_floats));
        if (!ws) return 1;
        if (qa.ws_floats > 0) use_workspace(qa, ws);
        if (qb.ws_floats > 0) use_workspace(qb, ws + first);
    }
    if (qa.best && qb.best && qa.best->groups > 1 && qb.best->groups > 1 &&
        gemm_fast_64x64k4_pairs(qa.la, qa.lb, qa.red, qb.la, qb.lb, qb.red)) {
        const char *label = "gemm_conv_backward";
        if (prof_enabled())
            label = prof_label("%s M=%d+%d J=%d+%d R=%d+%ld tile=%s split=%d+%d", label, a.M, b.M, a.J, b.J, a.R,
                               (long)b.R * b.nb, qa.best->name, qa.g.nsplit, qb.g.nsplit);
        {
            LaunchScope scope(label, product_flops(qa) + product_flops(qb), 0.0);
            if (gemm_fast_64x64k4_pair(qa.g, qb.g, qb.lb, s)) return 1;
        }
        if (check_launch(a.tag)) return 1;
    } else if (run_product(qa, s) || run_product(qb, s)) {
        return 1;
    }
    if (qa.ws_floats == 0 && qb.ws_floats == 0) return 0;
    ReduceJob ja, jb;
    double bytes = 0;
    if (qa.ws_floats > 0) bytes += reduce_job(qa, ja);
    if (qb.ws_floats > 0) bytes += reduce_job(qb, jb);
    if (qb.ws_floats == 0) return run_reduce(ja, bytes, s);
    if (qa.ws_floats == 0) return run_reduce(jb, bytes, s);
    {
        LaunchScope scope("gemm_split_reduce", 0.0, bytes);
        hipLaunchKernelGGL(split_reduce_pair_kernel, dim3(ja.blocks + jb.blocks), dim3(256), 0, s, ja, jb);
    }
    return check_launch("gemm_split_reduce");
}

}  // namespace thgpu

using namespace thgpu;

namespace {

// Column-major BLAS arguments as a GemmProblem.  Returns 1 for the quick returns of the reference
// dispatcher (nothing to do), -1 for a dimension the kernels cannot index, -2 for a null operand, 0 otherwise.
int blas_problem(GemmProblem &p, char transa, char transb, long m, long n, long k, float alpha, const float *a,
                 long lda, const float *b, long ldb, float beta, float *c, long ldc) {
    const bool ta = (transa == 't' || transa == 'T');
    const bool tb = (transb == 't' || transb == 'T');
    // Quick returns of the reference dispatcher (gputorch/lib/THC/THCBlas.cpp:257).
    if (!m || !n || ((alpha == 0 || !k) && beta == 1)) return 1;
    // Degenerate leading dimensions as TH fixes them up (TH/generic/THBlas.c:275-298).
    if (n == 1) ldc = m;
    if (ta) {
        if (m == 1) lda = k;
    } else {
        if (k == 1) lda = m;
    }
    if (tb) {
        if (k == 1) ldb = n;
    } else {
        if (n == 1) ldb = k;
    }
    if (m < 0 || n < 0 || k < 0 || m >= (1L << 31) || n >= (1L << 31) || k >= (1L << 31)) return -1;
    // a product that will touch memory needs its operands: a null pointer here would fault on the GPU
    if (!c || (alpha != 0 && k > 0 && (!a || !b))) return -2;
    // Column-major C(m x n) is the row-major n x m matrix C'(i', j') =
    // c[j' + i'*ldc]; C' = op(B)' * op(A)' with
    //   A'(i', r) = op(B)(r, i'),  B'(r, j') = op(A)(j', r).
    p.A = b;
    p.B = a;
    p.C = c;
    p.M = (int)n;
    p.J = (int)m;
    p.R = alpha == 0 ? 0 : (int)k;  // empty sum: C = beta*C, whatever A and B hold
    p.N = (int)m;
    p.a_rc = !tb;  // 'n': b[r + i'*ldb]
    p.sA = ldb;
    p.b_rc = ta;  // 't': a[r + j'*lda]
    p.sB = lda;
    p.sC = ldc;
    p.alpha = alpha;
    p.beta = beta;
    p.tag = "gemm_blas";
    return 0;
}

}  // namespace

extern "C" void THGPUBlas_gemm(char transa, char transb, long m, long n, long k, float alpha, float *a, long lda,
                               float *b, long ldb, float beta, float *c, long ldc) {
    GemmProblem p;
    const int rc = blas_problem(p, transa, transb, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc);
    if (rc > 0) return;
    if (rc < 0) {
        raise(rc == -2 ? "THGPUBlas_gemm: null operand" : "THGPUBlas_gemm: dimension exceeds 2^31");
        return;
    }
    if (gemm_launch(p)) raise("%s", thgpu_last_error());
}

extern "C" int thgpu_gemm_noalloc(char transa, char transb, long m, long n, long k, float alpha, const float *a,
                                  long lda, const float *b, long ldb, float beta, float *c, long ldc) {
    // Nothing here may allocate, so neither may a lazy initialisation: the stream and the address of the
    // static array exist only after thgpu_init.
    size_t cap = 0;
    float *ws = static_scratch(&cap);
    if (!ws) return fail("thgpu_gemm_noalloc: call thgpu_init() first (this entry point sets nothing up itself)");
    // (dimensions are range-checked before they are multiplied)
    if (m >= (1L << 31) || n >= (1L << 31) || k >= (1L << 31))
        return fail("thgpu_gemm_noalloc: dimension exceeds 2^31");
    if (m > 0 && n > 0 && m * n > (long)cap)
        return fail("thgpu_gemm_noalloc: a result of %ld x %ld elements exceeds the limit of %zu elements (%zu MiB)", m,
                    n, cap, cap * sizeof(float) >> 20);
    GemmProblem p;
    const int rc = blas_problem(p, transa, transb, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc);
    if (rc > 0) return 0;
    if (rc < 0) return fail(rc == -2 ? "thgpu_gemm_noalloc: null operand" : "thgpu_gemm_noalloc: dimension exceeds 2^31");
    p.ws_fixed = ws;
    p.ws_fixed_floats = (long)cap;
    p.tag = "gemm_blas_noalloc";
    return gemm_launch(p);
}

extern "C" int thgpu_gemm_strided_batched(char transa, char transb, long m, long n, long k, float alpha, const float *a,
                                          long lda, long stride_a, const float *b, long ldb, long stride_b, float beta,
                                          float *c, long ldc, long stride_c, long batch) {
    const bool ta = (transa == 't' || transa == 'T');
    const bool tb = (transb == 't' || transb == 'T');
    if (batch <= 0 || !m || !n) return 0;
    if (m >= (1L << 31) || n >= (1L << 31) || k >= (1L << 31)) return fail("gemm_strided_batched: dimension exceeds 2^31");
    if (stride_c == 0 && batch > 1) return fail("gemm_strided_batched: the results of a batch must not overlap");
    if (!c || (alpha != 0 && k > 0 && (!a || !b))) return fail("gemm_strided_batched: null operand");
    // One launch for the whole batch when op(B) is shared, op(A) = A and the batch's columns fit the
    // kernel's 32-bit tile indexing: the batch index then simply extends the columns of the (row-major,
    // transposed) product, as in the convolution's forward and gradInput GEMMs.
    if (!ta && stride_b == 0 && batch > 1 && m * batch < (1L << 31) && n * m * batch < (1L << 31)) {
        GemmProblem p;
        p.A = b;
        p.B = a;
        p.C = c;
        p.M = (int)n;
        p.J = (int)(m * batch);
        p.R = alpha == 0 ? 0 : (int)k;
        p.N = (int)m;
        p.a_rc = !tb;
        p.sA = ldb;
        p.b_rc = false;
        p.sB = lda;
        p.sC = ldc;
        p.bsB = stride_a;
        p.bsC = stride_c;
        p.alpha = alpha;
        p.beta = beta;
        p.tag = "gemm_blas_batched";
        return gemm_launch(p);
    }
    for (long i = 0; i < batch; ++i) {
        GemmProblem p;
        p.A = b + i * stride_b;
        p.B = a + i * stride_a;
        p.C = c + i * stride_c;
        p.M = (int)n;
        p.J = (int)m;
        p.R = alpha == 0 ? 0 : (int)k;
        p.N = (int)m;
        p.a_rc = !tb;
        p.sA = ldb;
        p.b_rc = ta;
        p.sB = lda;
        p.sC = ldc;
        p.alpha = alpha;
        p.beta = beta;
        p.tag = "gemm_blas_batched";
        if (gemm_launch(p)) return 1;
    }
    return 0;
}
