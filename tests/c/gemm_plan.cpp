// The planner of the GEMM calls (csrc/q4_gemm_plan.h) on the host: its estimates of the pipelined kernel
// against a schedule that hands out every workgroup, the choice for one weight, and what planning a call takes.
//   gemm_plan            prints "schedule ok", "choices ok", "widths ok", "rows ok", "pairs ok", "order ok" and, a line a call, its name and microseconds
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <queue>
#include <random>
#include <vector>

#include "q4_gemm_plan.h"

using namespace mi355q;

constexpr uint32_t kCus = 256;

// Every workgroup in turn to the compute unit that is free first; what is left when the first one has
// nothing more to do goes at the speed of a partly filled chip.
static double scheduled_us(const Variant &c, const GroupWork &work)
{
    std::priority_queue<double, std::vector<double>, std::greater<double>> free;
    for (uint32_t unit = 0; unit < kCus; ++unit) free.push(0.0);
    double groups = 0.0, steps = 0.0;
    for (uint32_t t = 0; t < work.count; ++t)
        for (uint64_t i = 0; i < work.groups[t]; ++i) {
            const double start = free.top();
            free.pop();
            free.push(start + c.fill + work.steps[t] * c.step);
            groups += 1.0;
            steps += work.steps[t];
        }
    const double first = free.top(), each = steps / groups;
    double last = first, busy = 0.0;
    for (; !free.empty(); free.pop()) {
        last = free.top();
        busy += last - first;
    }
    if (last - first < 1e-6) return first;
    const double r = busy / ((last - first) * kCus);
    return first + (last - first) *
                       (each * (c.part_step[0] + c.part_step[1] * std::fmax(0.0, r - 0.5)) + c.part_fill[0] + c.part_fill[1] * r * r) /
                       (each * c.step + c.fill);
}

static int check_schedules()
{
    std::mt19937 random(1);
    auto below = [&](uint32_t limit) { return (uint32_t)(random() % limit); };
    for (int round = 0; round < 400; ++round)
        for (int v = kFirstPiped; v < kVariants; ++v) {
            GroupWork work = {};
            work.count = 1u + below(kMaxTargets);
            uint32_t steps = 8u + below(80u);
            for (uint32_t t = 0; t < work.count; ++t) {
                work.steps[t] = steps;
                work.groups[t] = round % 5 == 0 ? kCus * (1u + below(3u)) : 1u + below(1200u);
                if (below(2u)) steps = 1u + below(steps);
            }
            const double expected = scheduled_us(variants[v], work);
            const double got = pipe_group_us(variants[v], kCus, work);
            if (std::fabs(got - expected) > 1e-6 * expected) {
                printf("shape %d, %u targets: %.6f, scheduled %.6f\n", v, work.count, got, expected);
                return 1;
            }
            work.count = 1;
            const double one = pipe_kernel_us(variants[v], kCus, work.groups[0], work.steps[0]);
            if (std::fabs(one - scheduled_us(variants[v], work)) > 1e-6 * one) {
                printf("shape %d, %u workgroups of %u steps: %.6f, scheduled %.6f\n", v, (unsigned)work.groups[0], work.steps[0], one,
                       scheduled_us(variants[v], work));
                return 1;
            }
        }
    printf("schedule ok\n");
    return 0;
}

struct Call {
    std::vector<Q4Device> weights;
    Q4LinearArgs a;
    Call(uint32_t M, uint32_t K, const std::vector<uint32_t> &widths) : weights(widths.size())
    {
        memset(&a, 0, sizeof a);
        a.M = M;
        a.count = (uint32_t)widths.size();
        for (size_t t = 0; t < widths.size(); ++t) {
            memset(&weights[t], 0, sizeof weights[t]);
            weights[t].N = widths[t];
            weights[t].K = K;
            weights[t].NT = (widths[t] + kTileRows - 1u) / kTileRows;
            weights[t].T = (K + kStepColumns - 1u) / kStepColumns;
            a.targets[t].w = &weights[t];
        }
    }
    Call(const Call &) = delete;
};

// The plan of a weight is what that weight alone is estimated to be fastest with, of every shape and split; only a
// weight of up to 48 steps that takes more than half of the chip in one round of the pipelined kernel may go
// without a split, as the fastest shape that does, for up to 12 % more.
static int check_choices(const mi355q_context *ctx)
{
    std::mt19937 random(2);
    for (int round = 0; round < 4000; ++round) {
        const uint32_t N = round == 0 ? 13312u : 64u + (uint32_t)(random() % 17408u), T = round == 0 ? 63u : 4u + (uint32_t)(random() % 132u);
        const uint32_t M = round == 0 ? 351u : 129u + (uint32_t)(random() % 1000u);
        Call call(M, T * kStepColumns, {N});
        const TargetPlan plan = plan_target(ctx, call.a, 0, M);
        for (int v = 0; v < kBytesVariant; ++v)
            for (uint32_t want = 1; want <= 8u && want * 8u <= T + 7u; ++want) {
                const Variant &c = variants[v];
                const uint32_t tpb = 4u * c.ntw + c.extra, n_blocks = (call.weights[0].NT + tpb - 1u) / tpb;
                const uint32_t steps = (T + want - 1u) / want, splits = (T + steps - 1u) / steps;
                const uint64_t groups = (uint64_t)n_blocks * ((M + c.bm - 1u) / c.bm) * splits;
                Around around = {};
                around.splits = splits;
                around.sums = splits > 1u ? (double)splits * M * N * 4e-6 : 0.0;
                around.outputs = (double)M * N * 2e-6;
                around.rows = (double)M * call.weights[0].K * 2e-6;
                around.reread = std::fmax(around.rows - 4.0, 0.0) * n_blocks;
                double us = launch_us(c, v >= kFirstPiped ? pipe_kernel_us(c, kCus, groups, steps)
                                                          : first_kernel_us(c, kCus, groups, steps), around);
                if (N % 4u != 0u) us += splits == 1u ? narrow_us(c, kCus, MI355Q_F16, groups) : kNarrowSumUs * M * N;
                const uint32_t blocks = (call.weights[0].NT + 15u) / 16u * ((M + 127u) / 128u);
                const bool whole = plan.splits == 1u && splits > 1u && T <= 48u && 2u * blocks > kCus && blocks <= kCus;
                if (us * (whole ? 1.12 : 1.0) < plan.us * (1.0 - 1e-9)) {
                    printf("%u x %u at %u rows: shape %d, %u splits, %.2f us; shape %d, %u splits is estimated at %.2f\n", N,
                           call.weights[0].K, M, plan.variant, plan.splits, plan.us, v, want, us);
                    return 1;
                }
            }
    }
    printf("choices ok\n");
    return 0;
}

// Outputs that the pipelined kernel and the kernel that adds K splits store one by one (a width that is no
// multiple of 4) count: 10212 columns take the first without a split, 3064 a split, two columns less or more neither.
static int check_widths(const mi355q_context *ctx)
{
    const struct { uint32_t M, K, N; } calls[] = {{440, 2688, 10212}, {440, 2688, 10214}, {345, 2560, 3064}, {345, 2560, 3062}};
    for (const auto &of : calls) {
        Call call(of.M, of.K, {of.N});
        const TargetPlan plan = plan_target(ctx, call.a, 0, of.M);
        if ((plan.variant >= kFirstPiped || plan.splits > 1u) != (of.N % 4u == 0u)) {
            printf("%u columns: shape %d, %u splits\n", of.N, plan.variant, plan.splits);
            return 1;
        }
    }
    printf("widths ok\n");
    return 0;
}

// One weight at 17 to 128 rows takes the kernel that was timed faster for it, q4_rows_kernel or another (us, weights from
// HBM), and two large ones at 32 rows the width of block that was.
static int check_rows(const mi355q_context *ctx)
{
    const struct { uint32_t M, K, N; int x; bool by_rows; } calls[] = {
        {36, 2944, 2928, MI355Q_F32, true},     // 16.1 by q4_rows_kernel, 17.1 by the other
        {28, 5120, 1280, MI355Q_F32, true},     // 14.8, 16.7
        {80, 5376, 14336, MI355Q_F16, true},    // 22.9, 33.0
        {84, 5312, 13758, MI355Q_F16, true},    // 25.6, 33.4
        {96, 5376, 14336, MI355Q_BF16, true},   // 30.4, 35.6
        {112, 5376, 14336, MI355Q_F16, false},  // 38.1, 33.7
        {112, 5120, 17408, MI355Q_F16, false},  // 41.0, 36.8
        {128, 6144, 5120, MI355Q_F16, false},   // 25.4, 21.3
        {100, 3584, 1024, MI355Q_F16, false},   // 12.7, 11.5
        {32, 6144, 5120, MI355Q_F16, true},     // 14.6, 14.8
        {32, 17408, 5120, MI355Q_F16, true},    // 22.5, 27.3
        {67, 17408, 5120, MI355Q_F16, true},    // 28.7, 35.8
        {67, 5120, 17408, MI355Q_F16, true},    // 29.0, 33.1
        {48, 2048, 1024, MI355Q_F16, true},     // 9.7, 11.6
        {36, 1152, 12000, MI355Q_BF16, true}};  // 11.8, 16.1
    for (const auto &of : calls) {
        Call call(of.M, of.K, {of.N});
        call.a.x_dtype = of.x;
        call.a.y_dtype = of.x;
        TargetPlan plans[kMaxTargets];
        GroupPlan group;
        RowsPlan rows;
        if (plan_gemm(ctx, call.a, plans, group, rows) != of.by_rows) {
            printf("%u x %u at %u rows of type %d: the other kernel\n", of.N, of.K, of.M, of.x);
            return 1;
        }
    }
    Call pair(32, 5120, {17408, 17408});  // 128 columns a block 33.0 us, 256 31.5
    TargetPlan plans[kMaxTargets];
    GroupPlan group;
    RowsPlan rows;
    if (!plan_gemm(ctx, pair.a, plans, group, rows) || rows.tiles != 16) {
        printf("two of 17408 x 5120 at 32 rows: %d tiles a block\n", rows.tiles);
        return 1;
    }
    printf("rows ok\n");
    return 0;
}

// fp32 calls of 65 rows and more: the weights of a call take q4_rows_kernel together or not at all, up to four times the columns
// of x, so that such a call is one launch; and the launch is not estimated to take longer than theirs, but for the estimates' own error.
static int check_pairs(const mi355q_context *ctx)
{
    std::mt19937 random(3);
    for (int round = 0; round < 6000; ++round) {
        const uint32_t T = 1u + (uint32_t)(random() % 18u), K = T * kStepColumns, M = 65u + (uint32_t)(random() % (round % 2 ? 200u : 1500u));
        std::vector<uint32_t> widths(1 + random() % kMaxTargets);
        for (uint32_t &N : widths) N = round == 0 ? 128u : 1u + (uint32_t)(random() % (4u * K));
        Call call(M, K, widths);
        call.a.x_dtype = call.a.y_dtype = call.a.residual_dtype = MI355Q_F32;
        TargetPlan plans[kMaxTargets];
        GroupPlan group;
        RowsPlan rows, other;
        bool taken[kMaxTargets];
        const uint32_t count = plan_pairs(ctx, call.a, taken, rows);
        if (count != 0u && count != call.a.count) {
            printf("%u of %u weights at %u rows of %u\n", count, call.a.count, M, K);
            return 1;
        }
        if (count == 0u) continue;
        plan_gemm(ctx, call.a, plans, group, other);
        double outputs = 0.0;
        for (const uint32_t N : widths) outputs += (double)M * N;
        const double us = rows_launch_us(kCus, T, outputs, rows) + 0.107e-6 * outputs * 4.0 + 3.24 + 1.86e-6 * 2.0 * M * K * 2.0;
        if (us > 1.1 * group.us) {
            printf("%u weights at %u rows of %u: %.1f us, as one launch of the others %.1f\n", call.a.count, M, K, us, group.us);
            return 1;
        }
    }
    printf("pairs ok\n");
    return 0;
}

// Weights that share a launch go out one by one under option "gemm_order", whose two orders are one weight's.
static int check_order(mi355q_context *ctx)
{
    Call call(512, 5120, {6144, 1024, 1024});
    for (const int order : {-1, 0, 1}) {
        ctx->gemm_order = order;
        TargetPlan plans[kMaxTargets];
        GroupPlan group;
        RowsPlan rows;
        if (plan_gemm(ctx, call.a, plans, group, rows) || (group.variant >= 0) != (order < 0)) {
            printf("order %d: shape %d for the weights together\n", order, group.variant);
            return 1;
        }
    }
    ctx->gemm_order = -1;
    printf("order ok\n");
    return 0;
}

static double planning_us(const mi355q_context *ctx, uint32_t M, uint32_t K, const std::vector<uint32_t> &widths)
{
    Call call(M, K, widths);
    const Q4LinearArgs &a = call.a;
    constexpr int kCalls = 200;
    double best = 1e30;
    volatile uint32_t sink = 0;
    for (int repeat = 0; repeat < 50; ++repeat) {
        const auto start = std::chrono::steady_clock::now();
        for (int i = 0; i < kCalls; ++i) {
            TargetPlan plans[kMaxTargets];
            GroupPlan group;
            RowsPlan rows;
            sink = sink + (plan_gemm(ctx, a, plans, group, rows) ? rows.units : plans[0].splits);
        }
        best = std::fmin(best, std::chrono::duration<double>(std::chrono::steady_clock::now() - start).count() * 1e6 / kCalls);
    }
    return best;
}

int main()
{
    if (check_schedules() != 0) return 1;
    mi355q_context *const ctx = (mi355q_context *)calloc(1, sizeof(mi355q_context));  // no device: what the planner reads
    if (ctx == nullptr) return 1;
    ctx->props.multiProcessorCount = (int)kCus;
    ctx->gemm_order = -1;
    if (check_choices(ctx) != 0 || check_widths(ctx) != 0 || check_rows(ctx) != 0 || check_pairs(ctx) != 0 || check_order(ctx) != 0) return 1;
    printf("q_k_v_32_rows %.2f\n", planning_us(ctx, 32, 5120, {6144, 1024, 1024}));
    printf("q_k_v_512_rows %.2f\n", planning_us(ctx, 512, 5120, {6144, 1024, 1024}));
    printf("gate_up_512_rows %.2f\n", planning_us(ctx, 512, 5120, {17408, 17408}));
    printf("down_512_rows %.2f\n", planning_us(ctx, 512, 17408, {5120}));
    free(ctx);
    return 0;
}
