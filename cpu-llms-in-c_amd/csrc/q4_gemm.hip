// Prefill GEMM on affine-Q4 weights: y[M][N] = x[M][K] * w[N][K]^T for M > 16.
// MFMA-bound.  The reference's batched kernels dequantize a weight tile to half
// precision and multiply it with 8x8 simdgroup MMAs, accumulating in fp32
// (qwen38_prefill.metal:953-1078,1373-1502; minimax_h3_attention.metal:211-592);
// its scalar check rounds the weight to fp16 the same way
// (minimax_h3_m3_gemm.m:87-104).  Here: w16 = fp16(s*q + b) (one fused fp16
// multiply-add per weight), fp16 x fp16 products on v_mfma_f32_16x16x32_f16,
// fp32 accumulation over the whole of K.
//
// Work split: a workgroup of four waves computes BM (64 or 128) rows of x by
// 4*NTW (+1) tiles of 16 rows of w.  The activations of one 128-column step are
// staged in LDS by LDS-direct loads (double buffered) and shared by the four
// waves; every wave dequantizes the codes of its own NTW tiles straight into the
// B-operand registers of the matrix instruction (the stream-tile layout hands
// each lane exactly the eight consecutive columns the instruction wants), so
// each weight is dequantized once per workgroup and never passes through LDS.
// The metadata is read as fp16 {scale, bias} pairs (converted at prepare for
// bf16 images).  Three kernels:
//   q4_gemm_kernel: two workgroups per compute unit overlap each other's
//     dequantization and matrix instructions (six tile shapes);
//   q4_gemm_pipe_kernel: one workgroup per compute unit, software pipelined by
//     hand (128 rows x 16, 17 or 20 tiles);
//   q4_rows_kernel (q4_rows_device.h): up to 128 rows, all weights of a call as
//     one launch; of fp32 activations also up to 256, in blocks of 16 to 64 rows' pairs.
// The host picks shape and K split by a time estimate fitted on this GPU (q4_gemm_plan.h), e.g.
// 20 tiles for the 17408-row matrices: 55 x 4 = 220 workgroups at M = 512.
// Several weights of a call go out as one launch where that is estimated to take less: they
// fill the chip together (us, a launch each -> one launch: 6144 + 1024 + 1024 x 5120 at 200 rows
// 51 -> 35, at 512 rows 78 -> 53; 2048 + 512 + 512 x 1024 at 512 rows 26.5 -> 10.5; two of
// 17408 x 5120 at 200 rows 106 -> 74; two of 8192 x 3072 at 512 rows 68 -> 43; three of 1280 x 1280
// over 1500 fp32 rows 72 -> 51).
#include <algorithm>
#include <cstdio>
#include "device_util.h"
#include "internal.h"

#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <utility>

#include "q4_gemm_plan.h"

namespace mi355q {

// the pipelined kernel's instantiations live in q4_gemm_pipe_*.hip
extern template __global__ void q4_gemm_pipe_kernel<128, 4, false, false>(const GemmGroup);
extern template __global__ void q4_gemm_pipe_kernel<128, 4, true, false>(const GemmGroup);
extern template __global__ void q4_gemm_pipe_kernel<128, 4, true, true>(const GemmGroup);
extern template __global__ void q4_gemm_pipe_kernel<128, 5, false, false>(const GemmGroup);
extern template __global__ void q4_gemm_pipe_kernel<128, 4, false, false, true>(const GemmParams);  // 8-bit codes
extern template __global__ void q4_gemm_pipe_kernel<128, 3, true, false, true>(const GemmParams);   // 8-bit codes

// Adds the K splits in split order (a fixed order) and applies the epilogue.  WIDE: a thread
// takes four adjacent outputs of one row (N a multiple of 4, y 16-byte aligned): 16-byte loads
// of each split's partial sums and one store; the additions are the same, in the same order.
//
// Activations that are not fp16 get the streaming kernel's treatment (q4_convert_x_launch): every
// row scaled by a power of two into fp16's range, bf16 rows as one fp16 row, fp32 rows as two
// (value, rounding remainder).  The matrix kernels multiply those M or 2 M rows; whoever holds the
// finished sums - their epilogue, or this kernel behind a K split - adds the two rows of a pair,
// takes the row's scale out again, adds the residual and converts.  (The reference's grouped
// linear keeps fp32 activations at any row count, whisper_turbo_encoder.c:128-176;
// cpu_q4_dot_float, qwen38_m3_layer.m:375-393.)
// A workgroup takes 256 (1024) adjacent columns of one output row: no index is ever divided (a
// division per thread cost the 27B prefill step's reductions about a microsecond each).
constexpr uint32_t kReduceThreads = 256;
constexpr uint32_t kReduceRows = 65535;  // of the grid's y; its z counts on

// Columns n (.. n + 3) of output row m from `splits` partial sums (SPLITS of them when that is not 0).
template <bool WIDE, int SPLITS>
__device__ __forceinline__ void reduce_columns(const GemmParams &p, uint32_t splits, uint32_t m, uint32_t n)
{
    typedef std::conditional_t<WIDE, floatx4, float> Piece;
    const uint32_t columns = padded_columns(p.N);
    const size_t stride = (size_t)p.M * columns;
    auto add = [](Piece &sum, const Piece &more) {
        if constexpr (WIDE) {
#pragma unroll
            for (int j = 0; j < 4; ++j) sum[j] += more[j];
        } else {
            sum += more;
        }
    };
    auto add_splits = [&](size_t from) {
        Piece sum = {};
        if constexpr (SPLITS > 0) {
            Piece piece[SPLITS];
#pragma unroll
            for (int s = 0; s < SPLITS; ++s) piece[s] = *(const Piece *)(p.partials + s * stride + from);
#pragma unroll
            for (int s = 0; s < SPLITS; ++s) add(sum, piece[s]);
        } else {
            for (uint32_t s = 0; s < splits; s += 4u) {  // four on their way at once; past the last it is read again
                Piece piece[4];
#pragma unroll
                for (uint32_t i = 0; i < 4u; ++i)
                    piece[i] = *(const Piece *)(p.partials + (s + i < splits ? s + i : splits - 1u) * stride + from);
#pragma unroll
                for (uint32_t i = 0; i < 4u; ++i)
                    if (s + i < splits) add(sum, piece[i]);
            }
        }
        return sum;
    };
    Piece value;
    if (p.pair) {
        value = add_splits((size_t)(2u * m) * columns + n);
        add(value, add_splits((size_t)(2u * m + 1u) * columns + n));
    } else {
        value = add_splits((size_t)m * columns + n);
    }
    if constexpr (WIDE) {
        finish_four(p, m, n, value);
    } else {
        const size_t at = (size_t)m * p.N + n;
        if (p.row_scale) value *= p.row_scale[m];
        if (p.residual) value += load_as_float(p.residual, p.residual_dtype, p.residual_is_bias ? n : at);
        store_from_float(p.y, p.y_dtype, at, value);
    }
}

// One target of a K split into at most eight: the number of splits is the host's, and all their
// loads are on their way before the first is added.  Launched behind every K split, a few
// microseconds of which the arguments' way is a good part: they are one cache line, read at once
// (ReduceParams), and fp16 activations (CONVERTED false) have no code for pairs and row scales.
// With the GEMM's own parameters and a loop over gridDim.y the arguments came in three round
// trips, one after the other (GEMM and sum, us: 5216 x 2752 at 96 rows 15.0 -> 14.3, 8192 x 3200 at
// 67 rows 18.0 -> 17.5, 6144 x 5120 at 200 rows 28.6 -> 28.0; the sum alone of 10000 columns at 200
// rows 5.2 -> 4.6, of 5120 at 512 rows from five 11.3 -> 10.5).
struct ReduceParams {
    const float *partials;
    void *y;
    const void *residual;
    const float *row_scale;
    uint32_t M, N;
    uint8_t y_dtype, residual_dtype, residual_is_bias, pair;
};
static_assert(sizeof(ReduceParams) <= 64, "one cache line of arguments");
template <bool WIDE, int SPLITS, bool CONVERTED>
__global__ void __launch_bounds__(kReduceThreads) q4_gemm_reduce_kernel(const ReduceParams of)
{
    GemmParams p = {};
    p.partials = const_cast<float *>(of.partials);
    p.y = of.y;
    p.residual = of.residual;
    p.M = of.M;
    p.N = of.N;
    p.y_dtype = of.y_dtype;
    p.residual_dtype = of.residual_dtype;
    p.residual_is_bias = of.residual_is_bias;
    p.wide_stores = WIDE;
    if constexpr (CONVERTED) {
        p.row_scale = of.row_scale;
        p.pair = of.pair;
    }
    const uint32_t n = (blockIdx.x * kReduceThreads + threadIdx.x) * (WIDE ? 4u : 1u);
    const uint32_t m = blockIdx.z * kReduceRows + blockIdx.y;
    if (n >= p.N || m >= (p.pair ? p.M / 2u : p.M)) return;
    reduce_columns<WIDE, SPLITS>(p, SPLITS, m, n);
}

// Every other sum: a loop over the splits, a call's targets, and the workgroups that share a
// column's block of q4_rows_kernel counted here.
template <bool WIDE>
__global__ void __launch_bounds__(kReduceThreads) q4_group_reduce_kernel(const GemmGroup group)
{
    uint32_t block = blockIdx.x;
    const GemmParams p = select_target<true>(group, block);
    const uint32_t n = (block * kReduceThreads + threadIdx.x) * (WIDE ? 4u : 1u);
    const uint32_t m = blockIdx.z * kReduceRows + blockIdx.y;
    if (n >= p.N || m >= (p.pair ? p.M / 2u : p.M)) return;
    uint32_t splits = p.splits;
    if (p.units) {
        const uint32_t begin = (p.first_block + n / p.block_columns) * p.T;
        splits = (begin + p.T - 1u) / p.units - begin / p.units + 1u;
    }
    if (splits == 1u) return;  // the outputs are stored: by one workgroup alone, of a target without a K split
    reduce_columns<WIDE, 0>(p, splits, m, n);
}

template <int BM, int NTW, bool EXTRA>
static hipError_t launch_gemm(mi355q_context *ctx, dim3 grid, const GemmGroup &group)
{
    const GemmParams &p = group.shared;
    if (p.targets > 1u)
        return p.row_scale ? launch(ctx, q4_gemm_group_kernel<BM, NTW, EXTRA, true>, grid, dim3(256), 0, group)
                           : launch(ctx, q4_gemm_group_kernel<BM, NTW, EXTRA, false>, grid, dim3(256), 0, group);
    return p.row_scale ? launch(ctx, q4_gemm_kernel<BM, NTW, EXTRA, true>, grid, dim3(256), 0, p)
                       : launch(ctx, q4_gemm_kernel<BM, NTW, EXTRA, false>, grid, dim3(256), 0, p);
}

// The pipelined kernel's stage is larger than the 64 KiB a kernel gets without asking: the
// limit is raised once per device and instantiation.
template <int NTW, bool XT>
static hipError_t launch_pipe(mi355q_context *ctx, dim3 grid, const GemmGroup &group)
{
    constexpr size_t bytes = pipe_lds_bytes(128);
    constexpr int slot = 2 * NTW + (XT ? 1 : 0);  // this instantiation's flag in the context
    static_assert(slot < 16, "mi355q_context::lds_raised holds sixteen flags");
    // per context (a context belongs to one device and serialises its calls): no process-wide
    // state, so contexts on different threads do not meet here; raising the limit twice is harmless
    if (!ctx->lds_raised[slot]) {
        hipError_t status = hipFuncSetAttribute((const void *)q4_gemm_pipe_kernel<128, NTW, XT>,
                                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (status != hipSuccess) return status;
        ctx->lds_raised[slot] = true;
    }
    return launch(ctx, q4_gemm_pipe_kernel<128, NTW, XT>, grid, dim3(256), bytes, group);
}

// The shapes on 8-bit codes: 16 tiles, or 13 (three per wave and one shared).
template <int NTW, bool XT>
static hipError_t launch_pipe_bytes(mi355q_context *ctx, dim3 grid, const GemmGroup &group)
{
    constexpr size_t bytes = pipe_lds_bytes(128);
    constexpr int slot = XT ? 13 : 14;
    if (!ctx->lds_raised[slot]) {
        hipError_t status = hipFuncSetAttribute((const void *)q4_gemm_pipe_kernel<128, NTW, XT, false, true>,
                                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (status != hipSuccess) return status;
        ctx->lds_raised[slot] = true;
    }
    return launch(ctx, q4_gemm_pipe_kernel<128, NTW, XT, false, true>, grid, dim3(256), bytes, group.shared);
}

// The 17-tile shape with compiler-managed weight loads (option "gemm_loads" = "plain").
static hipError_t launch_pipe_plain(mi355q_context *ctx, dim3 grid, const GemmGroup &group)
{
    constexpr size_t bytes = pipe_lds_bytes(128);
    constexpr int slot = 15;
    if (!ctx->lds_raised[slot]) {
        hipError_t status = hipFuncSetAttribute((const void *)q4_gemm_pipe_kernel<128, 4, true, true>,
                                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (status != hipSuccess) return status;
        ctx->lds_raised[slot] = true;
    }
    return launch(ctx, q4_gemm_pipe_kernel<128, 4, true, true>, grid, dim3(256), bytes, group);
}

// Adds the K splits of a launch's targets.
static hipError_t launch_reduce(mi355q_context *ctx, GemmGroup &group)
{
    bool wide = true;
    for (uint32_t t = 0; t < group.shared.targets; ++t) wide = wide && group.target[t].wide_stores;
    const uint32_t columns = kReduceThreads * (wide ? 4u : 1u);
    const GemmParams &p = group.shared;
    uint32_t blocks = 0;
    for (uint32_t t = 0; t < group.shared.targets; ++t) {
        group.target[t].first_reduce = blocks;
        if (p.units != 0u || group.target[t].splits > 1u) blocks += (group.target[t].N + columns - 1u) / columns;
    }
    const uint32_t rows = p.pair ? p.M / 2u : p.M;
    const dim3 grid(blocks, std::min(rows, kReduceRows), (rows + kReduceRows - 1u) / kReduceRows);
    if (p.targets != 1u || p.units != 0u || p.splits > 8u)  // (more than eight: only when forced)
        return wide ? launch(ctx, q4_group_reduce_kernel<true>, grid, dim3(kReduceThreads), 0, group)
                    : launch(ctx, q4_group_reduce_kernel<false>, grid, dim3(kReduceThreads), 0, group);
    const GemmTarget &target = group.target[0];
    const ReduceParams one = {target.partials, target.y, target.residual, p.row_scale, p.M, target.N, (uint8_t)p.y_dtype,
                              (uint8_t)p.residual_dtype, (uint8_t)(p.residual_is_bias != 0), (uint8_t)(p.pair != 0)};
    auto of = [&](auto splits) {
        constexpr int SPLITS = decltype(splits)::value;
        if (p.row_scale)
            return wide ? launch(ctx, q4_gemm_reduce_kernel<true, SPLITS, true>, grid, dim3(kReduceThreads), 0, one)
                        : launch(ctx, q4_gemm_reduce_kernel<false, SPLITS, true>, grid, dim3(kReduceThreads), 0, one);
        return wide ? launch(ctx, q4_gemm_reduce_kernel<true, SPLITS, false>, grid, dim3(kReduceThreads), 0, one)
                    : launch(ctx, q4_gemm_reduce_kernel<false, SPLITS, false>, grid, dim3(kReduceThreads), 0, one);
    };
    switch (p.splits) {
    case 2: return of(std::integral_constant<int, 2>());
    case 3: return of(std::integral_constant<int, 3>());
    case 4: return of(std::integral_constant<int, 4>());
    case 5: return of(std::integral_constant<int, 5>());
    case 6: return of(std::integral_constant<int, 6>());
    case 7: return of(std::integral_constant<int, 7>());
    default: return of(std::integral_constant<int, 8>());
    }
}

// Rows, row scales and pairs of the activations the matrix kernels see: x itself when it is fp16,
// else its conversion in the context's staging buffer (made here when `convert`: the targets of
// one call share it): M rows, or 2 M when fp32 activations go in as (value, remainder) pairs.
static int gemm_activations(mi355q_context *ctx, const Q4LinearArgs &a, uint32_t x_columns, bool convert, GemmParams &p,
                            char *error, size_t error_capacity)
{
    p.pair = a.x_dtype == MI355Q_F32;
    p.M = p.pair ? 2u * a.M : a.M;
    p.x = (const _Float16 *)a.x;
    if (a.x_dtype == MI355Q_F16) return MI355Q_OK;
    // [ the rows' inverse scales, padded to 256 bytes | rows * K fp16 ]
    const size_t scale_bytes = ((size_t)a.M * sizeof(float) + 255u) & ~(size_t)255u;
    int status = ensure_stage(ctx, 3, scale_bytes + (size_t)p.M * x_columns * sizeof(_Float16), error, error_capacity);
    if (status != MI355Q_OK) return status;
    float *const scales = (float *)ctx->stage[3];
    _Float16 *const fp16_rows = (_Float16 *)((char *)ctx->stage[3] + scale_bytes);
    if (convert) {
        hipError_t converted = q4_convert_x_launch(ctx, a.x, a.x_dtype, fp16_rows, scales, a.M, x_columns);
        if (converted != hipSuccess) return fail_hip(converted, "activation conversion launch", error, error_capacity);
    }
    p.x = fp16_rows;
    p.row_scale = scales;
    return MI355Q_OK;
}

// Targets first .. first + count - 1 of a call in one launch: the shape `variant`, each target with the
// K split of its own plan; `convert`: the call's activations have not been converted yet.
static int gemm_targets(mi355q_context *ctx, const Q4LinearArgs &a, uint32_t first, uint32_t count, const TargetPlan *plans,
                        int variant, bool convert, char *error, size_t error_capacity)
{
    const Q4Device &shape = *a.targets[first].w;  // columns and kind are the same for all
    const bool bytes_kernel = plans[first].bytes;
    if (a.x_columns != 0 && (a.x_columns * 2u != shape.K || a.x_columns % kStepColumns != 0)) {
        set_error(error, error_capacity, "q4 gemm: a repeated activation row is half the weight's columns, whole 128-column steps");
        return MI355Q_ERROR_INVALID;
    }
    const uint32_t x_columns = a.x_columns ? a.x_columns : shape.K;
    GemmGroup group;
    memset(&group, 0, sizeof group);
    GemmParams &p = group.shared;
    int status = gemm_activations(ctx, a, x_columns, convert, p, error, error_capacity);
    if (status != MI355Q_OK) return status;
    const Variant &chosen = variants[variant];
    const uint32_t tpb = 4u * chosen.ntw + chosen.extra;
    const uint32_t rows = p.M, m_blocks = (rows + chosen.bm - 1) / chosen.bm;
    p.K = x_columns;
    p.T = bytes_kernel ? shape.T / 2u : shape.T;
    p.wrap_steps = a.x_columns && !bytes_kernel ? a.x_columns / kStepColumns : 0xffffffffu;
    p.y_dtype = a.y_dtype;
    p.residual_dtype = a.residual_dtype;
    p.residual_is_bias = a.residual_is_bias;
    p.targets = count;
    size_t sums = 0;  // floats of partial sums
    bool split = false;
    for (uint32_t t = 0; t < count; ++t) {
        const Q4Device &w = *a.targets[first + t].w;
        GemmTarget &target = group.target[t];
        target.codes = bytes_kernel ? w.codes8 : w.codes;
        target.meta = bytes_kernel ? w.meta8 : w.meta16;  // fp16 {scale, bias}: the weight is evaluated in fp16 here
        target.y = a.targets[first + t].y;
        target.residual = a.targets[first + t].residual;
        target.N = w.N;
        target.NT = w.NT;
        target.wide_stores = w.N % 4u == 0u && (uintptr_t)target.y % 16u == 0u;
        target.steps_per_split = (p.T + plans[first + t].splits - 1) / plans[first + t].splits;
        target.splits = (p.T + target.steps_per_split - 1) / target.steps_per_split;
        if (target.splits > 1u) {
            split = true;
            sums += (size_t)target.splits * rows * padded_columns(w.N);
        }
        if (ctx->trace)
            fprintf(stderr, "mi355q: q4 gemm M=%u N=%u K=%u -> variant %d (BM=%d, %d tiles/wave%s%s), K split %u%s\n",
                    rows, w.N, w.K, variant, chosen.bm, chosen.ntw, chosen.extra ? " +1" : "",
                    bytes_kernel ? ", 8-bit codes" : "", target.splits, t ? ", same launch" : "");
    }
    if (split) {
        status = ensure_stage(ctx, 4, sums * sizeof(float), error, error_capacity);
        if (status != MI355Q_OK) return status;
    }
    // the longest first: what is left to start late is short
    std::stable_sort(group.target, group.target + count,
                     [](const GemmTarget &l, const GemmTarget &r) { return l.steps_per_split > r.steps_per_split; });
    float *partials = (float *)ctx->stage[4];
    uint32_t blocks = 0;
    for (uint32_t t = 0; t < count; ++t) {
        GemmTarget &target = group.target[t];
        const uint32_t n_blocks = (target.NT + tpb - 1) / tpb;
        target.first_block = blocks;
        blocks += (n_blocks * m_blocks * target.splits + 7u) / 8u * 8u;
        if (target.splits > 1u) {
            target.partials = partials;
            partials += (size_t)target.splits * rows * padded_columns(target.N);
        }
    }
    dim3 grid(blocks);
    if (count == 1u) {
        const GemmTarget &target = group.target[0];
        p.codes = target.codes;
        p.meta = target.meta;
        p.y = target.y;
        p.residual = target.residual;
        p.partials = target.partials;
        p.N = target.N;
        p.NT = target.NT;
        p.wide_stores = target.wide_stores;
        p.splits = target.splits;
        p.steps_per_split = target.steps_per_split;
        // Workgroups go to the XCDs in turn: when the number of tile blocks is a multiple of eight, the
        // row blocks of one tile block already meet on one XCD and read their weights through one L2;
        // otherwise the pipelined kernel renumbers its blocks so that they do (2-3 % on the 100-block
        // 8-bit gate, about 1 % on the 20-block down projection, nothing or slightly worse where the
        // launch order was already right).  With K splits the renumbering also gives every XCD one
        // split's columns of the activations instead of all of them (down at M = 512: 193 -> 86 MB
        // fetched, 0.7 % faster).
        const uint32_t n_blocks = (target.NT + tpb - 1) / tpb;
        p.xcd_order = ctx->gemm_order >= 0 ? ctx->gemm_order
                                           : ((n_blocks % 8u != 0u && m_blocks > 1u) || p.splits > 1u ? 1 : 0);
        grid = dim3(n_blocks, m_blocks, p.splits);
    }
    hipError_t launched = hipErrorInvalidValue;
    switch (variant) {
    case 0: launched = launch_gemm<128, 4, false>(ctx, grid, group); break;
    case 1: launched = launch_gemm<128, 2, false>(ctx, grid, group); break;
    case 2: launched = launch_gemm<64, 4, false>(ctx, grid, group); break;
    case 3: launched = launch_gemm<64, 4, true>(ctx, grid, group); break;
    case 4: launched = launch_gemm<64, 2, false>(ctx, grid, group); break;
    case 5: launched = launch_gemm<64, 2, true>(ctx, grid, group); break;
    case 6: launched = launch_pipe<4, false>(ctx, grid, group); break;
    case 7: launched = ctx->gemm_plain_loads ? launch_pipe_plain(ctx, grid, group) : launch_pipe<4, true>(ctx, grid, group); break;
    case 8: launched = launch_pipe<5, false>(ctx, grid, group); break;
    case 9: launched = launch_pipe_bytes<4, false>(ctx, grid, group); break;
    default: launched = launch_pipe_bytes<3, true>(ctx, grid, group); break;
    }
    if (launched != hipSuccess)
        return fail_hip(launched, "q4 gemm kernel launch", error, error_capacity);
    if (split) {
        launched = launch_reduce(ctx, group);
        if (launched != hipSuccess)
            return fail_hip(launched, "q4 gemm reduce launch", error, error_capacity);
    }
    return MI355Q_OK;
}

// ---- 17..128 rows: q4_rows_kernel (q4_rows_device.h) ---------------------------------------

static int q4_rows_linears(mi355q_context *ctx, const Q4LinearArgs &a, const RowsPlan &plan, char *error,
                           size_t error_capacity)
{
    const Q4Device &first = *a.targets[0].w;
    if (a.x_columns != 0 && (a.x_columns * 2u != first.K || a.x_columns % kStepColumns != 0)) {
        set_error(error, error_capacity, "q4 gemm: a repeated activation row is half the weight's columns, whole 128-column steps");
        return MI355Q_ERROR_INVALID;
    }
    const uint32_t x_columns = a.x_columns ? a.x_columns : first.K;
    GemmGroup group;
    memset(&group, 0, sizeof group);
    GemmParams &p = group.shared;
    int status = gemm_activations(ctx, a, x_columns, true, p, error, error_capacity);
    if (status != MI355Q_OK) return status;
    p.M = a.M;  // the kernel adds the sums of value and remainder rows itself
    p.pair = 0;
    p.m_blocks = plan.m_blocks;
    p.K = x_columns;
    p.T = first.T;
    p.wrap_steps = a.x_columns ? a.x_columns / kStepColumns : 0xffffffffu;
    p.y_dtype = a.y_dtype;
    p.residual_dtype = a.residual_dtype;
    p.residual_is_bias = a.residual_is_bias;
    p.splits = 1;
    p.units = plan.units;
    p.total_units = plan.blocks * p.T;
    p.block_columns = (uint32_t)plan.tiles * kTileRows;
    p.targets = a.count;
    // blocks are shared unless every workgroup takes whole ones; a block meets at most this many
    const bool sharing = p.units % p.T != 0u && p.units < p.total_units;
    const uint32_t sharers = (p.T - 1u) / p.units + 2u;
    if (sharing) {
        size_t columns = 0;
        for (uint32_t t = 0; t < a.count; ++t) columns += padded_columns(a.targets[t].w->N);
        status = ensure_stage(ctx, 4, (size_t)sharers * p.M * columns * sizeof(float), error, error_capacity);
        if (status != MI355Q_OK) return status;
    }
    float *partials = (float *)ctx->stage[4];
    uint32_t blocks = 0;
    for (uint32_t t = 0; t < a.count; ++t) {
        const Q4Device &w = *a.targets[t].w;
        GemmTarget &target = group.target[t];
        target.codes = w.codes;
        target.meta = w.meta16;
        target.y = a.targets[t].y;
        target.residual = a.targets[t].residual;
        target.N = w.N;
        target.NT = w.NT;
        target.wide_stores = w.N % 4u == 0u && (uintptr_t)target.y % 16u == 0u;
        target.first_block = blocks;
        blocks += (w.NT + plan.tiles - 1u) / plan.tiles * plan.m_blocks;
        if (sharing) {
            target.partials = partials;
            partials += (size_t)sharers * p.M * padded_columns(w.N);
        }
    }
    const uint32_t groups = (p.total_units + p.units - 1u) / p.units;
    if (ctx->trace)
        fprintf(stderr, "mi355q: q4 rows M=%u K=%u -> %d fragments%s x %u columns, %u workgroups, %u steps each\n", p.M, p.K,
                plan.mf, plan.pair ? " of pairs" : "", p.block_columns, groups, p.units);
    hipError_t launched = plan.tiles == 4    ? q4_rows_launch_4(ctx, plan.mf, plan.pair, groups, group)
                          : plan.tiles == 8  ? q4_rows_launch_8(ctx, plan.mf, plan.pair, groups, group)
                                             : q4_rows_launch_16(ctx, plan.mf, plan.pair, groups, group);
    if (launched != hipSuccess) return fail_hip(launched, "q4 rows kernel launch", error, error_capacity);
    if (sharing) {
        launched = launch_reduce(ctx, group);
        if (launched != hipSuccess) return fail_hip(launched, "q4 gemm reduce launch", error, error_capacity);
    }
    return MI355Q_OK;
}

// Whether no target of the call writes what another one reads or writes, nor the activations:
// only then may they run at the same time (and share converted activations).
static bool targets_independent(const Q4LinearArgs &a)
{
    auto overlap = [](const void *p, size_t p_bytes, const void *q, size_t q_bytes) {
        return (uintptr_t)p < (uintptr_t)q + q_bytes && (uintptr_t)q < (uintptr_t)p + p_bytes;
    };
    const size_t x_bytes = (size_t)a.M * (a.x_columns ? a.x_columns : a.targets[0].w->K) * dtype_bytes(a.x_dtype);
    for (uint32_t t = 0; t < a.count; ++t) {
        const size_t y_bytes = (size_t)a.M * a.targets[t].w->N * dtype_bytes(a.y_dtype);
        if (overlap(a.targets[t].y, y_bytes, a.x, x_bytes)) return false;
        for (uint32_t u = 0; u < a.count; ++u) {
            if (u == t) continue;
            const size_t cells = (a.residual_is_bias ? 1u : (size_t)a.M) * a.targets[u].w->N;
            if (overlap(a.targets[t].y, y_bytes, a.targets[u].y, (size_t)a.M * a.targets[u].w->N * dtype_bytes(a.y_dtype)))
                return false;
            if (a.targets[u].residual != nullptr &&
                overlap(a.targets[t].y, y_bytes, a.targets[u].residual, cells * dtype_bytes(a.residual_dtype)))
                return false;
        }
    }
    return true;
}

int q4_gemm_linears(mi355q_context *ctx, const Q4LinearArgs &a, char *error, size_t error_capacity)
{
    int status = MI355Q_OK;
    if (a.count > 1u && !targets_independent(a)) {  // one after the other, in the caller's order
        for (uint32_t t = 0; t < a.count && status == MI355Q_OK; ++t) {
            Q4LinearArgs one = a;
            one.count = 1;
            one.targets[0] = a.targets[t];
            status = q4_gemm_linears(ctx, one, error, error_capacity);
        }
        return status;
    }
    TargetPlan plans[kMaxTargets];
    RowsPlan together;
    GroupPlan group;
    bool taken[kMaxTargets];
    const uint32_t pairs = plan_pairs(ctx, a, taken, together);
    if (pairs == a.count) return q4_rows_linears(ctx, a, together, error, error_capacity);
    Q4LinearArgs rest = a;
    if (pairs != 0u) {  // those targets by q4_rows_kernel, the others behind them on the same converted activations
        Q4LinearArgs part = a;
        part.count = rest.count = 0;
        for (uint32_t t = 0; t < a.count; ++t) {
            Q4LinearArgs &to = taken[t] ? part : rest;
            to.targets[to.count++] = a.targets[t];
        }
        status = q4_rows_linears(ctx, part, together, error, error_capacity);
        if (status != MI355Q_OK) return status;
    }
    if (plan_gemm(ctx, rest, plans, group, together)) return q4_rows_linears(ctx, rest, together, error, error_capacity);
    const bool convert = pairs == 0u;
    if (group.variant >= 0)
        return gemm_targets(ctx, rest, 0, rest.count, plans, group.variant, convert, error, error_capacity);
    for (uint32_t t = 0; t < rest.count && status == MI355Q_OK; ++t)
        status = gemm_targets(ctx, rest, t, 1, plans, plans[t].variant, convert && t == 0u, error, error_capacity);
    return status;
}

}  // namespace mi355q
