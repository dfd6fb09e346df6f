// How a call of the GEMM kernels goes out: shapes, K splits, launches.  Host code that runs on every call before
// its first launch: on one core, us, a 27B layer's q|k|v at 32 and at 512 rows 0.9 and 0.8, gate|up 0.5, down 0.4
// (the K splits of one weight estimated like a launch of several, whose workgroups take compute units in turn:
// 7.9, 7.2, 4.8, 3.5).
#pragma once
#include <algorithm>

#include "internal.h"
#include "q4_rows_device.h"

namespace mi355q {

// The shapes, and what a launch of each is estimated to take: microseconds of a call among others, fitted
// to timings on this GPU of one weight under every shape and K split (27 weights from 896 x 3584 to
// 17408 x 5120 at 75 to 4646 rows, ten of them at 17 to 128, six 8-bit weights; 210 to 1130 timings a
// shape, 4 to 5 % rms).  The shape and split that the estimates choose takes 0.7 % longer than the best
// timed one of these on average, 11 % at most (estimates that left out what launches, K splits' second kernels
// and stores take: 3 %, 26 %); of 178 random calls above 128 rows that nothing was fitted to 1.3 %, 19 % at
// most, and four above 10 %.
struct Variant {
    int bm, ntw, extra;
    int resident;           // workgroups that fit one compute unit (registers, LDS)
    double launch;          // once
    double step, fill;      // a chip full of workgroups: each 128-column step, and once
    // First kernel: the same of a chip with at most k + 1 workgroups on a compute unit, which the
    // last workgroups are.  Pipelined kernel, whose last round of workgroups takes the fraction r of
    // the compute units: {step, + max(0, r - 0.5) of each step}, {fill, + r^2} (the chip is power
    // limited, and up to about half of it the clock stays near its maximum).
    double part_step[4], part_fill[4];
    double split, per_split, sums;  // a K split: its second kernel, more for each split, MB of partial sums
    double outputs;         // MB of outputs
    double converted[3];    // activations that are not fp16: once, MB of fp16 rows, MB of outputs
    double reread;          // MB of fp16 rows beyond an XCD's L2, by each block of tiles
    // Pipelined kernel without a K split, outputs whose width is no multiple of 4 and which it stores one by one:
    // a round of the chip with fp16, fp32, bf16 activations.  (One more column than 10208, 4096, 14336 by 2688, 4096,
    // 5120 at 440, 300, 700 rows; 25 and 12 more of 8-bit codes.  Left out, 10214 x 2688 at 440 rows took 45.6 us in a
    // shape estimated at 39, where one of the first kernel takes 34, and 23677 8-bit x 1728 at 154 rows 58 instead of 46.)
    double narrow[3];
};
constexpr Variant variants[] = {
    {128, 4, 0, 2, 13.19, 3.208, 5.98, {2.167, 3.026}, {0.0, 1.16}, 0.0, 0.0, 0.192, 0.435, {2.27, 0.36, 0.0}, 0.000, {}},
    {128, 2, 0, 2, 5.82, 1.628, 0.0, {1.207, 1.595}, {0.0, 0.010}, 2.52, 0.0, 0.304, 0.474, {5.72, 0.40, 0.046}, 0.007, {}},
    {64, 4, 0, 3, 5.54, 2.755, 0.0, {1.175, 1.820, 2.868}, {0.53, 0.0, 0.0}, 2.60, 0.0, 0.262, 0.566, {5.81, 0.27, 0.0}, 0.000, {}},
    {64, 4, 1, 2, 8.64, 2.275, 0.0, {1.366, 2.151}, {0.037, 0.0}, 1.82, 0.0, 0.250, 0.206, {3.96, 0.29, 0.31}, 0.002, {}},
    {64, 2, 0, 4, 4.16, 1.831, 0.0, {0.711, 1.054, 1.516, 1.972}, {0.41, 1.14, 0.61, 0.0}, 2.52, 0.0, 0.280, 0.498, {4.84, 0.37, 0.0}, 0.003, {}},
    {64, 2, 1, 2, 4.99, 1.240, 0.0, {0.918, 1.294}, {0.0, 0.21}, 2.46, 0.0, 0.279, 0.524, {4.76, 0.36, 0.21}, 0.000, {}},
    {128, 4, 0, 1, 4.51, 1.363, 5.31, {1.107, 0.117}, {3.93, 2.92}, 2.48, 0.24, 0.207, 0.325, {5.48, 0.18, 0.50}, 0.014, {10.8, 3.7, 13.5}},
    {128, 4, 1, 1, 6.29, 1.545, 6.04, {1.260, 0.291}, {3.64, 1.55}, 2.40, 0.32, 0.182, 0.355, {5.22, 0.19, 0.56}, 0.011, {12.4, 4.2, 16.0}},
    {128, 5, 0, 1, 1.25, 1.747, 6.38, {1.368, 0.627}, {9.07, 0.22}, 2.98, 0.28, 0.175, 0.363, {5.14, 0.23, 0.50}, 0.003, {15.5, 5.3, 18.7}},
    // 16 and 13 tiles on 8-bit codes, and only for them
    {128, 4, 0, 1, 0.88, 1.544, 9.49, {1.249, 0.535}, {5.21, 6.69}, 4.14, 0.10, 0.172, 0.031, {0.0, 0.0, 0.0}, 0.000, {10.0, 3.5, 13.4}},
    {128, 3, 1, 1, 5.81, 1.436, 6.56, {1.144, 0.482}, {0.0, 4.74}, 4.30, 0.14, 0.208, 0.054, {0.0, 0.0, 0.0}, 0.000, {9.8, 2.4, 10.0}}};
constexpr int kVariants = sizeof variants / sizeof variants[0];
constexpr int kFirstPiped = 6;    // the first shape of the pipelined kernel
constexpr int kBytesVariant = 9;  // the first on 8-bit codes

// the pipelined kernel addresses x with 32-bit byte offsets and whole 128-column steps
inline bool gemm_pipe_ok(const Q4Device &w, uint32_t rows, uint32_t x_columns)
{
    return w.K % kStepColumns == 0 && (uint64_t)rows * x_columns * sizeof(_Float16) + 16384u < (1ull << 32);
}

// What a launch takes besides its matrix kernel.
struct Around {
    uint32_t splits;       // the most of one target
    double sums, outputs;  // MB
    double rows;           // MB of fp16 rows
    double reread;         // MB
    bool converted;
};
inline double launch_us(const Variant &c, double kernel_us, const Around &around)
{
    double us = c.launch + kernel_us;
    if (around.splits > 1u) us += c.split + c.per_split * around.splits + c.sums * around.sums;
    if (around.converted) us += c.converted[0] + c.converted[1] * around.rows + c.converted[2] * around.outputs;
    return us + c.outputs * around.outputs + c.reread * around.reread;
}

// Microseconds of the first kernel, `each` steps a workgroup: full rounds of the chip, then what is left.
inline double first_kernel_us(const Variant &c, uint32_t cus, uint64_t groups, double each)
{
    const uint64_t slots = (uint64_t)cus * c.resident, rounds = groups < slots ? 0u : groups / slots;
    uint64_t rest = groups - rounds * slots;
    double us = (double)rounds * (each * c.step + c.fill);
    if (rest != 0u) {
        int k = 0;
        for (; rest > cus; rest -= cus) ++k;
        us += each * c.part_step[k] + c.part_fill[k];
    }
    return us;
}

// The last round of the pipelined kernel, on the fraction r of the compute units.
inline double pipe_rest_us(const Variant &c, double each, double r)
{
    return each * (c.part_step[0] + c.part_step[1] * std::max(0.0, r - 0.5)) + c.part_fill[0] + c.part_fill[1] * r * r;
}

// Microseconds of the pipelined kernel, one workgroup per compute unit: one target, whole rounds and a rest.
inline double pipe_kernel_us(const Variant &c, uint32_t cus, uint64_t groups, uint32_t steps)
{
    const uint64_t rounds = groups < cus ? 0u : groups / cus, rest = groups - rounds * cus;
    double us = (double)rounds * (c.fill + (double)steps * c.step);
    if (rest != 0u) us += pipe_rest_us(c, (double)steps, (double)rest / (double)cus);
    return us;
}

// Its stores of narrow outputs (Variant::narrow), beside that.
inline double narrow_us(const Variant &c, uint32_t cus, int x_dtype, uint64_t groups)
{
    const uint64_t rounds = groups <= cus ? groups != 0u : (groups + cus - 1u) / cus;
    return c.narrow[x_dtype == MI355Q_F16 ? 0 : x_dtype == MI355Q_F32 ? 1 : 2] * (double)rounds;
}

// What the kernel that adds K splits takes more for each narrow output, whose row it also stores one value at a time
// (10210, 4098, 14338 columns against four-column multiples at 150 to 700 rows: 0.5 to 5.5 us).
constexpr double kNarrowSumUs = 0.45e-6;

// What each target gives a launch of several, the longest workgroups first.
struct GroupWork {
    uint32_t count;
    uint32_t steps[kMaxTargets];   // of a workgroup
    uint64_t groups[kMaxTargets];
};

// The same of several targets: the workgroups take the compute units as they come free.
inline double pipe_group_us(const Variant &c, uint32_t cus, const GroupWork &work)
{
    struct Level {
        double at;  // so many compute units are free from here on
        uint64_t units;
    } level[kMaxTargets + 2];  // a target adds at most one
    int levels = 1;
    level[0] = {0.0, cus};
    uint64_t groups = 0, steps = 0;
    for (uint32_t i = 0; i < work.count; ++i) {
        const double time = c.fill + (double)work.steps[i] * c.step;
        uint64_t left = work.groups[i];
        groups += left;
        steps += left * work.steps[i];
        while (left > 0u) {
            if (levels == 1 && left >= cus) {  // whole rounds
                level[0].at += time * (double)(left / cus);
                left %= cus;
                continue;
            }
            const uint64_t taken = std::min(left, level[0].units);  // those that are free first
            const Level busy = {level[0].at + time, taken};
            left -= taken;
            level[0].units -= taken;
            if (level[0].units == 0u) {
                for (int l = 1; l < levels; ++l) level[l - 1] = level[l];
                --levels;
            }
            int at = levels;
            while (at > 0 && level[at - 1].at > busy.at + 1e-9) --at;
            if (at > 0 && level[at - 1].at > busy.at - 1e-9) {
                level[at - 1].units += taken;
            } else {
                for (int l = levels; l > at; --l) level[l] = level[l - 1];
                level[at] = busy;
                ++levels;
            }
        }
    }
    double us = level[0].at, busy = 0.0;  // busy: of all compute units together, from the first one's end on
    for (int l = 0; l < levels; ++l) busy += (level[l].at - level[0].at) * (double)level[l].units;
    const double rest = level[levels - 1].at - level[0].at;
    if (rest > 0.0) {
        const double r = busy / (rest * cus), each = (double)steps / (double)groups;
        us += rest * pipe_rest_us(c, each, r) / (each * c.step + c.fill);
    }
    return us;
}

// How one target of a call is multiplied: the shape and K split with the smallest estimated time.
struct TargetPlan {
    bool bytes;       // by the kernel for 8-bit codes
    int variant;
    uint32_t splits;
    double us;        // the estimate
};

// A target splits K the same way in company as alone, so that it has the same bits, and two weights that each
// take more than half of the chip fill it together, in one round of the pipelined kernel, without splits.
// Such a weight of up to 48 steps takes a split of the pipelined kernel only where that is estimated to gain
// 12 %.  Seventeen pairs were 30 % faster than as launches with splits of their own, us: two of 17408 x 5120 at 200
// rows 74 instead of 96, of 8368 x 5248 at 487 75 instead of 97.  The weight alone pays for it: up to a tenth of
// its time with the split (17408 x 5120 at 200 rows 52 instead of 50, 6144 x 6144 at 726 61 instead of 60).  From 52 steps on, and held back from
// splits of the first kernel, it pays more than a pair gains (13312 x 8064 at 351 rows 90 instead of 79, 5696 x
// 7424 at 687 77 instead of 65, 8512 x 8064 at 401 83 instead of 69).
constexpr double kSplitWeight = 1.12;
constexpr uint32_t kWholeSteps = 48;
inline TargetPlan plan_target(const mi355q_context *ctx, const Q4LinearArgs &a, uint32_t target, uint32_t rows)
{
    const Q4Device &w = *a.targets[target].w;
    const uint32_t x_columns = a.x_columns ? a.x_columns : w.K;
    // The doubled form of an 8-bit weight whose activation row the kernels would read twice: the
    // kernel for 8-bit codes reads the bytes themselves instead, one pass over the row, half the
    // matrix instructions.  It is the pipelined kernel, with that kernel's conditions.
    const bool bytes = w.codes8 != nullptr && a.x_columns != 0 && !ctx->q8_gemm_doubled &&
                       (uint64_t)rows * x_columns * sizeof(_Float16) + 16384u < (1ull << 32);
    const uint32_t T = bytes ? w.T / 2u : w.T;
    const bool pipe_ok = gemm_pipe_ok(w, rows, x_columns);
    TargetPlan best = {bytes, 0, 1, 1e30}, whole = best;  // whole: without a split
    // Decomposition: BM rows x (4*NTW + EXTRA) tiles per workgroup, K split in `splits`: up to eight, of eight
    // steps or so at least.
    uint32_t ways = 0, want[8], steps[8], splits[8];
    for (uint32_t s = 1; s <= 8u && s * 8u <= T + 7u; ++s) {
        const uint32_t of_steps = (T + s - 1u) / s;
        if (ways != 0u && of_steps == steps[ways - 1u]) continue;  // the split before it again
        want[ways] = s;
        steps[ways] = of_steps;
        splits[ways++] = (T + of_steps - 1u) / of_steps;
    }
    const uint32_t cus = (uint32_t)ctx->props.multiProcessorCount;
    Around around;
    around.outputs = (double)a.M * w.N * dtype_bytes(a.y_dtype) * 1e-6;
    around.converted = a.x_dtype != MI355Q_F16;
    around.rows = (double)rows * w.K * sizeof(_Float16) * 1e-6;
    const double sums = (double)rows * w.N * 4e-6;
    for (int v = bytes ? kBytesVariant : 0; v < (bytes ? kVariants : kBytesVariant); ++v) {
        if (v >= kFirstPiped && !pipe_ok) break;
        const Variant &c = variants[v];
        const uint32_t tpb = 4u * c.ntw + c.extra, n_blocks = (w.NT + tpb - 1u) / tpb;
        const uint64_t blocks = (uint64_t)n_blocks * ((rows + c.bm - 1u) / c.bm);
        around.reread = std::max(around.rows - 4.0, 0.0) * n_blocks;
        for (uint32_t i = 0; i < ways; ++i) {
            around.splits = splits[i];
            around.sums = splits[i] > 1u ? splits[i] * sums : 0.0;
            double us = launch_us(c, v >= kFirstPiped ? pipe_kernel_us(c, cus, blocks * splits[i], steps[i])
                                                      : first_kernel_us(c, cus, blocks * splits[i], steps[i]), around);
            if (w.N % 4u != 0u) us += splits[i] == 1u ? narrow_us(c, cus, a.x_dtype, blocks) : kNarrowSumUs * a.M * w.N;
            if (us < best.us) best = {bytes, v, want[i], us};
            if (i == 0u && us < whole.us) whole = {bytes, v, 1u, us};
        }
    }
    const uint64_t pipe_blocks = (uint64_t)((w.NT + 15u) / 16u) * ((rows + 127u) / 128u);  // of 128 rows x 16 tiles
    if (best.splits > 1u && best.variant >= kFirstPiped && !bytes && T <= kWholeSteps && 2u * pipe_blocks > cus &&
        pipe_blocks <= cus && whole.us < kSplitWeight * best.us)
        best = whole;
    // option "q4_gemm" = "VARIANT,SPLITS" for experiments
    if (ctx->force_gemm[1] >= 1 && ctx->force_gemm[0] < kVariants && (ctx->force_gemm[0] < kFirstPiped || pipe_ok) &&
        (ctx->force_gemm[0] >= kBytesVariant) == bytes) {
        best.variant = ctx->force_gemm[0];
        best.splits = (uint32_t)ctx->force_gemm[1];
    }
    return best;
}

// The targets above 128 rows: as one launch of one shape, or each by its own plan (variant -1).  In one
// launch, too, each has the K split of its own plan, and so its own call's bits.
struct GroupPlan {
    int variant;
    double us;
};
inline GroupPlan plan_group(const mi355q_context *ctx, const Q4LinearArgs &a, uint32_t rows, const TargetPlan *plans)
{
    GroupPlan best = {-1, 0.0};
    bool alike = a.count > 1u && ctx->gemm_order < 0;  // (an order asked for is that of a weight's own launch)
    for (uint32_t t = 0; t < a.count; ++t) {
        best.us += plans[t].us;
        if (t != 0u && a.x_dtype != MI355Q_F16) {  // one conversion serves them all
            const Variant &c = variants[plans[t].variant];
            best.us -= c.converted[0] + c.converted[1] * (double)rows * a.targets[t].w->K * sizeof(_Float16) * 1e-6;
        }
        alike = alike && !plans[t].bytes;  // (the kernel of 8-bit codes takes one target)
    }
    if (!alike) return best;
    if (ctx->force_gemm[1] >= 1) {
        if (plans[0].variant == ctx->force_gemm[0]) best.variant = plans[0].variant;
        return best;
    }
    const double alone_us = best.us;
    const Q4Device &first = *a.targets[0].w;
    const bool pipe_ok = gemm_pipe_ok(first, rows, a.x_columns ? a.x_columns : first.K);
    const uint32_t cus = (uint32_t)ctx->props.multiProcessorCount;
    GroupWork work = {};
    work.count = a.count;
    uint32_t splits[kMaxTargets], NT[kMaxTargets];
    bool odd[kMaxTargets];  // of a width that is no multiple of 4
    double narrow_sums = 0.0;
    Around around = {};
    around.converted = a.x_dtype != MI355Q_F16;
    around.rows = (double)rows * first.K * sizeof(_Float16) * 1e-6;
    for (uint32_t t = 0; t < a.count; ++t) {
        const Q4Device &w = *a.targets[t].w;
        const uint32_t steps = (first.T + plans[t].splits - 1u) / plans[t].splits, ways = (first.T + steps - 1u) / steps;
        around.splits = std::max(around.splits, ways);
        if (ways > 1u) around.sums += (double)ways * rows * w.N * 4e-6;
        around.outputs += (double)a.M * w.N * dtype_bytes(a.y_dtype) * 1e-6;
        if (w.N % 4u != 0u && ways > 1u) narrow_sums += kNarrowSumUs * a.M * w.N;
        uint32_t at = t;
        for (; at > 0u && work.steps[at - 1u] < steps; --at) {
            work.steps[at] = work.steps[at - 1u];
            splits[at] = splits[at - 1u];
            NT[at] = NT[at - 1u];
            odd[at] = odd[at - 1u];
        }
        work.steps[at] = steps;
        splits[at] = ways;
        NT[at] = w.NT;
        odd[at] = w.N % 4u != 0u;
    }
    for (int v = 0; v < kBytesVariant; ++v) {
        if (v >= kFirstPiped && !pipe_ok) break;
        const Variant &c = variants[v];
        const uint32_t tpb = 4u * c.ntw + c.extra, m_blocks = (rows + c.bm - 1u) / c.bm;
        uint64_t groups = 0, steps = 0, narrow = 0;
        around.reread = 0.0;
        for (uint32_t t = 0; t < a.count; ++t) {
            const uint32_t n_blocks = (NT[t] + tpb - 1u) / tpb;
            work.groups[t] = (uint64_t)n_blocks * m_blocks * splits[t];
            groups += work.groups[t];
            steps += work.groups[t] * work.steps[t];
            if (odd[t] && splits[t] == 1u) narrow += work.groups[t];
            around.reread += std::max(around.rows - 4.0, 0.0) * n_blocks;
        }
        const double us = launch_us(c, v >= kFirstPiped ? pipe_group_us(c, cus, work)
                                                        : first_kernel_us(c, cus, groups, (double)steps / (double)groups), around) +
                          narrow_us(c, cus, a.x_dtype, narrow) + narrow_sums;
        if (us < 0.95 * alone_us && us < best.us) best = {v, us};
    }
    return best;
}

// ---- 17..128 rows: q4_rows_kernel (q4_rows_device.h) ---------------------------------------

struct RowsPlan {
    int mf, tiles;                 // 16-row fragments of fp16 rows, tiles a block
    bool pair;                     // fp32 activations: pairs of fp16 rows
    uint32_t m_blocks;             // blocks of rows
    uint32_t blocks, units;        // blocks in all, units per workgroup
};

// The launch of q4_rows_kernel for a call's targets together; false: not the kernel for it.
// `others_us`: what they would take otherwise.
// Shape and workgroups minimise a microsecond estimate fitted to 14000 timings on this GPU (526 calls of one to three
// weights from 128 x 512 to two of 17408 x 5120, 9 to 64 rows of fp32, 17 to 128 of fp16 and bf16, every block width, whole
// blocks and 128 and 256 workgroups; each with weights from HBM, from the Infinity Cache, and between two large calls,
// where the chip runs slower; 5 % rms; the launch it chooses takes 0.5 % more than the best timed one on average): a
// unit's arithmetic, longer the more of the chip works (power), or its bytes; the end of every block in a workgroup's run,
// which is why runs that divide a block are worth more; where workgroups share blocks the second kernel and the partial
// sums; the conversion of activations that are not fp16; the outputs.  (Without the power and the ends: 1.3 %; two of
// 17408 x 5120 at 32 rows took 128 columns a block, 33.0 us, and not 256, 31.5.)
//
// It is taken up to 1.05 times the other kernels' estimate for several weights of up to 96 matrix rows, 0.98 times of more
// where they are large, and up to 0.89 times otherwise, 0.95 of 16-bit outputs of up to 64 rows: 0.1 to 0.7 % more time than
// with the better of the two, above 96 rows 1 to 2 % (us from HBM and between large calls, this kernel and the others:
// 14336 x 5376 at 67 rows 24.3 and 30.7, 21.5 and 29.4; 5120 x 6144 at 48 rows 15.4 and 16.0, 14.7 and 13.5; 17408 x 5120
// at 112 rows 41 and 37; 6144 + 1024 + 1024 x 5120 at 67 rows 18.0 and 26.2, 17.9 and 23.0; two of 3584 x 1024 at 128 rows
// from the Infinity Cache 10.8 and 9.9; two of 17408 x 5120 at 128 rows between large calls 61.5 and 65.4).
// A unit, by tiles a block (4, 8, 16) and fragments:
constexpr double kRowsUnitUs[3][9] = {{0, 0, 0.327, 0.380, 0.389, 0.434, 0.483, 0, 0.733},
                                      {0, 0, 0.425, 0.506, 0.622, 0.647, 0.733, 0, 0.971},
                                      {0, 0, 0.782, 0.873, 0.991, 1.123, 1.186, 0, 1.382}};

// A launch of T steps a block, without the conversion and the outputs.
inline double rows_launch_us(uint32_t cus, uint32_t T, double outputs, const RowsPlan &plan)
{
    const uint32_t total = plan.blocks * T, units = plan.units, groups = (total + units - 1u) / units;
    const uint32_t rounds = (groups + cus - 1u) / cus;
    const bool sharing = units % T != 0u && units < total;
    const double mf = plan.mf, tiles = plan.tiles, filled = (double)groups / ((double)rounds * cus);
    const double unit = std::max(kRowsUnitUs[plan.tiles / 8][plan.mf] * (1.0 + 0.0227 * mf * (filled - 0.75)),
                                 0.051 * tiles * filled + 0.0483 * mf);
    // ends of blocks in the longest run, and workgroups that share a block
    const double ends = !sharing ? std::max(1u, units / T) : T % units == 0u ? 1.0 : (units - 2u) / T + 2u;
    const double sharers = T % units == 0u ? T / units : (T + units - 1.0) / units;
    const double us = 3.78 + rounds * (units * unit + ends * (plan.pair ? 0.0119 : 0.0237) * mf * tiles);
    return sharing ? us + 3.21 + sharers * (0.0781 + 1.53e-6 * outputs) : us;
}

inline bool rows_plan(const mi355q_context *ctx, const Q4LinearArgs &a, uint32_t rows, double others_us, RowsPlan &plan)
{
    const Q4Device &first = *a.targets[0].w;
    const uint32_t T = first.T;
    if (rows > 128u) return false;
    // 8-bit weights with byte tiles have a kernel that reads those
    if (a.x_columns != 0 && first.codes8 != nullptr && !ctx->q8_gemm_doubled) return false;
    plan.pair = a.x_dtype == MI355Q_F32;
    plan.m_blocks = 1;
    plan.mf = (int)((a.M + 15u) / 16u) * (plan.pair ? 2 : 1);
    if (plan.mf < 2) plan.mf = 2;
    if (plan.mf == 7) plan.mf = 8;
    auto shape = [&](int tiles) {
        plan.tiles = tiles;
        plan.blocks = 0;
        for (uint32_t t = 0; t < a.count; ++t) plan.blocks += (a.targets[t].w->NT + tiles - 1u) / tiles;
        return (uint64_t)plan.blocks * T < (1ull << 31);
    };
    if (ctx->force_gemm[1] >= 1) {
        // option "q4_gemm": 11, 12, 13 = 4, 8, 16 tiles a block; 1 = whole blocks, s = 64 (s - 1) workgroups
        const int which = ctx->force_gemm[0];
        if (which < 11 || which > 13 || !shape(4 << (which - 11))) return false;
        const uint32_t groups = ctx->force_gemm[1] == 1 ? plan.blocks : 64u * (uint32_t)(ctx->force_gemm[1] - 1);
        plan.units = (plan.blocks * T + groups - 1u) / groups;
        return true;
    }
    const uint32_t cus = (uint32_t)ctx->props.multiProcessorCount;
    double outputs = 0.0, best_cost = 1e30;
    for (uint32_t t = 0; t < a.count; ++t) outputs += (double)a.M * a.targets[t].w->N;
    RowsPlan best = plan;
    for (const int tiles : {4, 8, 16}) {
        if (!shape(tiles)) return false;
        const uint32_t total = plan.blocks * T;
        for (const uint32_t want : {plan.blocks, cus / 2u, cus}) {
            plan.units = (total + want - 1u) / want;
            const double cost = rows_launch_us(cus, T, outputs, plan);
            if (cost < best_cost) {
                best_cost = cost;
                best = plan;
            }
        }
    }
    plan = best;
    best_cost += 0.107e-6 * outputs * dtype_bytes(a.y_dtype);
    if (a.x_dtype != MI355Q_F16) best_cost += 3.24 + 1.86e-6 * rows * first.K * sizeof(_Float16);
    double most = 0.89;
    if (a.count != 1u && (rows <= 96u || others_us > 20.0))
        most = rows <= 96u ? 1.05 : 0.98;
    else if (a.count == 1u && rows <= 64u && a.y_dtype != MI355Q_F32)
        most = 0.95;
    return best_cost <= most * others_us;
}

// ---- 65 to 256 rows of fp32: q4_rows_kernel on whole blocks of 16 to 64 rows' pairs ------------------------

// Weights of 3 to 14 steps, fp32 outputs.  The other kernels multiply value and remainder rows like rows of their own,
// in blocks whose fill and stores nothing hides (us, those and this kernel: three of 1280 x 1280 at 150 rows 21.9 and
// 14.0, 1280 x 1280 at 150 rows 15.5 and 11.6, 5120 x 1280 at 150 rows 17.0 and 15.1, 140 x 1280 at 203 rows 14.2 and 11.5).
// A weight has the bits of its own call in company, so it takes this kernel whatever shares the call: by the rows and
// columns of x, which the weights of a call have in common, and not by an estimate of its own call, which parted
// calls in two launches with a conversion each (2688 + 128 x 1280 at 319 rows 22 -> 33 us).  Weights more than four times as wide
// as x are left out (those of an encoder's or a decoder's layer are not as wide); a call that has both kinds is parted.
// More rows or wider weights fill the chip with the other kernels' larger blocks: calls whose outputs were more than 512 times
// the columns of x lost at times (28440 x 384 at 152 rows 20 -> 27, 5120 x 1280 at 1345 rows 55 -> 64).  Of more than 14 steps
// the others split K into more sums than this kernel's two, whose error is smaller.
constexpr uint32_t kPairsRows = 256, kPairsSteps[2] = {3, 14}, kPairsWide = 4;
inline bool pairs_take(const mi355q_context *ctx, const Q4LinearArgs &a, const Q4Device &w)
{
    if (a.x_dtype != MI355Q_F32 || a.M <= 64u || a.x_columns != 0u || w.K % kStepColumns != 0u || ctx->gemm_order >= 0) return false;
    if (ctx->force_gemm[1] >= 1)  // 32-bit offsets into a block's rows, and steps in all
        return ctx->force_gemm[0] >= 11 && ctx->force_gemm[0] <= 13 && (uint64_t)w.K * 256u < (1ull << 32) &&
               (uint64_t)(w.NT + 3u) / 4u * w.T * ((a.M + 15u) / 16u) * kMaxTargets < (1ull << 31);
    return a.y_dtype == MI355Q_F32 && a.residual_dtype == MI355Q_F32 && a.M <= kPairsRows && w.T >= kPairsSteps[0] &&
           w.T <= kPairsSteps[1] && w.N <= kPairsWide * w.K;
}

// The targets that it takes (their number) and the launch for them.  The block is chosen by the estimate above (0.2 % more time
// than the best timed one over 800 calls).  Outputs do not depend on it: in these forms two waves share a tile's columns.
inline uint32_t plan_pairs(const mi355q_context *ctx, const Q4LinearArgs &a, bool *taken, RowsPlan &plan)
{
    const uint32_t cus = (uint32_t)ctx->props.multiProcessorCount, T = a.targets[0].w->T;
    uint32_t count = 0;
    for (uint32_t t = 0; t < a.count; ++t) {
        taken[t] = pairs_take(ctx, a, *a.targets[t].w);
        if (taken[t]) ++count;
    }
    if (count == 0u) return 0;
    RowsPlan at;
    at.pair = true;
    auto shape = [&](int tiles, int mf) {
        at.tiles = tiles;
        at.mf = mf;
        at.m_blocks = (a.M + 8u * mf - 1u) / (8u * mf);
        at.blocks = 0;
        for (uint32_t t = 0; t < a.count; ++t)
            if (taken[t]) at.blocks += (a.targets[t].w->NT + tiles - 1u) / tiles * at.m_blocks;
        at.units = (at.blocks + cus - 1u) / cus * T;
        return mf * tiles <= 64;  // (else a wave takes whole columns)
    };
    if (ctx->force_gemm[1] >= 1) {
        // option "q4_gemm": 11, 12, 13 = 4, 8, 16 tiles a block; s = 1 .. 4 for 16 to 64 rows, 5 .. 8 for two blocks a workgroup, ...
        const int s = ctx->force_gemm[1] - 1;
        if (!shape(4 << (ctx->force_gemm[0] - 11), 2 * (s % 4 + 1))) return 0;
        at.units = std::min((uint32_t)s / 4u + 1u, at.blocks) * T;
        plan = at;
        return count;
    }
    double best = 1e30;
    for (const int tiles : {4, 8, 16})
        for (const int mf : {2, 4, 6, 8}) {
            if (!shape(tiles, mf)) continue;
            const double us = rows_launch_us(cus, T, 0.0, at);
            if (us < best) {
                best = us;
                plan = at;
            }
        }
    return count;
}

// The call: by q4_rows_kernel as `rows_launch` says (true), else by `group` and `plans`.
inline bool plan_gemm(const mi355q_context *ctx, const Q4LinearArgs &a, TargetPlan *plans, GroupPlan &group, RowsPlan &rows_launch)
{
    const uint32_t rows = a.x_dtype == MI355Q_F32 ? 2u * a.M : a.M;
    for (uint32_t t = 0; t < a.count; ++t) {
        uint32_t same = 0;  // gate and up, k and v: planned once
        while (same < t && (a.targets[same].w->N != a.targets[t].w->N || a.targets[same].w->codes8 != nullptr ||
                            a.targets[t].w->codes8 != nullptr))
            ++same;
        plans[t] = same < t ? plans[same] : plan_target(ctx, a, t, rows);
    }
    group = plan_group(ctx, a, rows, plans);
    return rows_plan(ctx, a, rows, group.us, rows_launch);
}

}  // namespace mi355q
