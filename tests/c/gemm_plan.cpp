// The planner of the GEMM calls (csrc/q4_gemm_plan.h) on the host: its estimates of the pipelined kernel
// against a schedule that hands out every workgroup, and what planning a call takes.
//   gemm_plan            prints "schedule ok" and, a line a call, its name and microseconds
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

static double planning_us(const mi355q_context *ctx, uint32_t M, uint32_t K, const std::vector<uint32_t> &widths)
{
    std::vector<Q4Device> weights(widths.size());
    Q4LinearArgs a;
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
    printf("q_k_v_32_rows %.2f\n", planning_us(ctx, 32, 5120, {6144, 1024, 1024}));
    printf("q_k_v_512_rows %.2f\n", planning_us(ctx, 512, 5120, {6144, 1024, 1024}));
    printf("gate_up_512_rows %.2f\n", planning_us(ctx, 512, 5120, {17408, 17408}));
    printf("down_512_rows %.2f\n", planning_us(ctx, 512, 17408, {5120}));
    free(ctx);
    return 0;
}
