// Device code of the affine-Q4 linear for 17..128 rows of x: more rows than the streaming kernel
// takes, too few to keep the matrix cores busy.  Bound by memory and by what a launch costs
// besides: the 27B gate|up pair is 100 MB of weights (16 us at the rate of a large copy) and
// 11 GFLOP at 32 rows (5 us).
#pragma once
#include "q4_gemm_device.h"

namespace mi355q {

// Loads that write LDS directly (uniform base + 32-bit lane offset); lane l's bytes land at
// lds_base + 16 l (4 l).  NT: use-once data.  m0 is named as clobbered so that the compiler
// carries no value of its own in it across the statement (it warns that m0 is reserved, which is
// the point).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <bool NT>
__device__ __forceinline__ void rows_load_x4(uint32_t lane_offset, const char *base, uint32_t lds_base)
{
    if constexpr (NT)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt"
                     :
                     : "v"(lane_offset), "s"(base), "s"(lds_base)
                     : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                     :
                     : "v"(lane_offset), "s"(base), "s"(lds_base)
                     : "memory", "m0");
}
__device__ __forceinline__ void rows_load_x1(uint32_t lane_offset, const char *base, uint32_t lds_base)
{
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                 :
                 : "v"(lane_offset), "s"(base), "s"(lds_base)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

// One stage = one 128-column step of a workgroup: 16 * MF rows of x (256 bytes each), then each of
// the four waves' own NTW tiles of codes, then their metadata.
constexpr uint32_t rows_stage_bytes(int mf, int ntw) { return (uint32_t)mf * 4096u + 4u * (uint32_t)ntw * 1024u + rows_meta_loads(ntw) * 1024u; }
// Stages in the ring: two workgroups on a compute unit when three stages each fit its 160 KiB (up
// to four), else one workgroup with up to five.
constexpr int rows_stages(int mf, int ntw)
{
    const int two = (int)(80u * 1024u / rows_stage_bytes(mf, ntw)), one = (int)(160u * 1024u / rows_stage_bytes(mf, ntw));
    return two >= 3 ? (two > 4 ? 4 : two) : one > 5 ? 5 : one;
}
constexpr uint32_t rows_lds_bytes(int mf, int ntw) { return (uint32_t)rows_stages(mf, ntw) * rows_stage_bytes(mf, ntw); }

// A workgroup of four waves: 16 * MF rows of x by 4 * NTW tiles of w (of one of the call's
// weights), a run of 128-column steps (K split over blockIdx.y; a second kernel adds the splits).
// Everything a step needs - the rows of x, shared by the waves, and each wave's own codes and
// metadata - is written to LDS by LDS-direct loads, so the steps in flight (two or three ahead of
// the arithmetic) cost no registers and one counted wait per step covers all of them: the loads
// are asm statements in one in-order queue that the compiler adds nothing to.  The weight is
// rounded as in the other GEMM kernels, w16 = fp16(s*q + b), and multiplied with the weights as
// the first operand: lane (r, kq) holds row 16*i + r, columns tile*16 + 4*kq .. + 3.
template <int MF, int NTW>
__global__ void __launch_bounds__(256, 2) q4_rows_kernel(const GemmGroup group)
{
    extern __shared__ uint4 rows_lds[];
    constexpr int TPB = 4 * NTW;
    constexpr int R = rows_stages(MF, NTW);
    constexpr int META = (int)rows_meta_loads(NTW);
    constexpr int S = MF + NTW + META;  // loads a wave puts in flight per step
    static_assert(R >= 3 && S * (R - 1) <= 63, "two steps ahead at least; the load counter has six bits");
    constexpr uint32_t STAGE = rows_stage_bytes(MF, NTW), CODES = MF * 4096u, METAS = CODES + TPB * 1024u;
    typedef __attribute__((address_space(3))) void *lds_ptr;

    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r = lane & 15u, kq = lane >> 4;
    uint32_t block;
    const GemmParams p = select_target(group, blockIdx.x, block);
    const uint32_t split = blockIdx.y;
    const uint32_t step_begin = split * p.steps_per_split;
    const uint32_t step_end = step_begin + p.steps_per_split < p.T ? step_begin + p.steps_per_split : p.T;
    const uint32_t count = step_end - step_begin;  // the host's splits are never empty
    const uint32_t tile0 = block * TPB + wave * NTW;

    // Lane offsets, fixed for the whole kernel.  Rows beyond M re-read the last row, tiles beyond
    // NT the last tile's codes and the last metadata word: in bounds, and never stored.
    uint32_t x_lane[MF], codes_lane[NTW], meta_lane[META];
#pragma unroll
    for (int j = 0; j < MF; ++j) {
        const uint32_t local = 4u * (MF * wave + j) + kq;
        const uint32_t m = local < p.M ? local : p.M - 1u;
        x_lane[j] = (m * p.K + 8u * (r ^ (local & 15u))) * (uint32_t)sizeof(_Float16);
    }
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
        const uint32_t tile = tile0 + t < p.NT ? tile0 + t : p.NT - 1u;
        codes_lane[t] = (tile * 64u + lane) * (uint32_t)sizeof(uint4);
    }
#pragma unroll
    for (int q = 0; q < META; ++q) {
        const uint32_t at = tile0 * 128u + q * 256u + lane * 4u, last = p.NT * 128u - 4u;
        meta_lane[q] = at < last ? at : last;
    }
    // when K is an odd multiple of 64 the upper half of the last step does not exist (its codes and
    // metadata are zero): such lanes read the lower half again, 64 columns back in their row
    const bool odd_tail = p.K % kStepColumns != 0u;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr)rows_lds);
    auto fetch = [&](uint32_t i, uint32_t slot) {
        const uint32_t step = step_begin + i, x_step = step >= p.wrap_steps ? step - p.wrap_steps : step;
        const char *const x_at = (const char *)(p.x + (size_t)x_step * kStepColumns);
        const char *const codes_at = (const char *)(p.codes + (size_t)step * p.NT * 64u);
        const char *const meta_at = (const char *)(p.meta + (size_t)step * p.NT * 16u);
        const uint32_t at = lds0 + slot * STAGE;
        const bool tail = odd_tail && step + 1u == p.T;
#pragma unroll
        for (int j = 0; j < MF; ++j) {
            const uint32_t octet = r ^ ((4u * (MF * wave + j) + kq) & 15u);
            const uint32_t offset = tail && octet >= 8u ? x_lane[j] - 128u : x_lane[j];
            rows_load_x4<false>(offset, x_at, at + (MF * wave + j) * 1024u);
        }
#pragma unroll
        for (int t = 0; t < NTW; ++t) rows_load_x4<true>(codes_lane[t], codes_at, at + CODES + (wave * NTW + t) * 1024u);
#pragma unroll
        for (int q = 0; q < META; ++q) rows_load_x1(meta_lane[q], meta_at, at + METAS + (wave * META + q) * 256u);
    };

    floatx4 acc[NTW][MF];
#pragma unroll
    for (int t = 0; t < NTW; ++t)
#pragma unroll
        for (int i = 0; i < MF; ++i) acc[t][i] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    const NibbleMasks masks = nibble_masks();

    static_for<R - 1>([&](auto i_c) {
        if ((uint32_t) decltype(i_c)::value < count) fetch(decltype(i_c)::value, decltype(i_c)::value);
    });
    uint32_t slot = 0;
    for (uint32_t i = 0; i < count; ++i) {
        // this wave's loads of step i have landed once only those of the younger steps are left
        const uint32_t younger = count - 1u - i;
        if (younger >= (uint32_t)(R - 2)) {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(S * (R - 2)) : "memory");
        } else {
            static_for<R - 2>([&](auto n_c) {
                if (younger == (uint32_t) decltype(n_c)::value)
                    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(S * decltype(n_c)::value) : "memory");
            });
        }
        // behind the barrier every wave's have, and every wave has read the last of step i - 1,
        // whose slot the fetch of step i + R - 1 fills
        asm volatile("s_barrier" ::: "memory");
        const uint32_t before = slot == 0u ? R - 1u : slot - 1u;
        if (i + R - 1u < count) fetch(i + R - 1u, before);

        const char *const stage = (const char *)rows_lds + slot * STAGE;
        uint4 codes[NTW];
        uint2 meta[NTW];
#pragma unroll
        for (int t = 0; t < NTW; ++t) {
            codes[t] = *(const uint4 *)(stage + CODES + (wave * NTW + t) * 1024u + lane * 16u);
            meta[t] = *(const uint2 *)(stage + METAS + wave * (META * 256u) + t * 128u + r * 8u);
        }
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            half8 x_frag[MF];
#pragma unroll
            for (int m = 0; m < MF; ++m)
                x_frag[m] = __builtin_bit_cast(half8, *(const uint4 *)(stage + (16u * m + r) * 256u + ((4u * d + kq) ^ r) * 16u));
#pragma unroll
            for (int t = 0; t < NTW; ++t) {
                half8 scale, bias;
                meta_to_half(d < 2 ? meta[t].x : meta[t].y, scale, bias);
                const uint32_t word = d == 0 ? codes[t].x : d == 1 ? codes[t].y : d == 2 ? codes[t].z : codes[t].w;
                const half8 w16 = dequant8(word, masks, scale, bias);
#pragma unroll
                for (int m = 0; m < MF; ++m)
                    acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w16, x_frag[m], acc[t][m], 0, 0, 0);
            }
        }
        slot = slot + 1u == R ? 0u : slot + 1u;
    }

#pragma unroll
    for (int t = 0; t < NTW; ++t) {
        const uint32_t n = (tile0 + t) * kTileRows + 4u * kq;
#pragma unroll
        for (int i = 0; i < MF; ++i) {
            floatx4 values = acc[t][i];
            uint32_t m = 16u * i + r;
            if (p.pair && p.splits <= 1u) {  // rows 2m and 2m + 1 are adjacent lanes
#pragma unroll
                for (int j = 0; j < 4; ++j) values[j] += __shfl_xor(values[j], 1, 64);
                if ((m & 1u) == 0u && m < p.M && n < p.N) finish_four(p, split, m >> 1, n, values);
                continue;
            }
            if (m < p.M && n < p.N) finish_four(p, split, m, n, values);
        }
    }
}

}  // namespace mi355q
