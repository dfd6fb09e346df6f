// Device code of the affine-Q4 linear for 17..128 rows of x: more rows than the streaming kernel
// takes, too few to keep the matrix cores busy.  Bound by memory and by what a launch costs
// besides: the 27B gate|up pair is 100 MB of weights (16 us at the rate of a large copy) and
// 11 GFLOP at 32 rows (5 us).
#pragma once
#include "q4_gemm_device.h"

namespace mi355q {

// One stage = one 128-column step of a workgroup: 16 * MF rows of x (256 bytes each), then each
// wave's own NTW tiles of codes, then their metadata.
constexpr uint32_t rows_stage_bytes(int mf, int ntw, int waves)
{
    return (uint32_t)mf * 4096u + (uint32_t)waves * ((uint32_t)ntw * 1024u + 256u);
}
// Stages in the ring: two workgroups on a compute unit when three stages each fit its 160 KiB (up
// to four), else one workgroup with what fits, three to five.
constexpr int rows_resident(int mf, int ntw, int waves) { return 3u * rows_stage_bytes(mf, ntw, waves) <= 80u * 1024u ? 2 : 1; }
constexpr int rows_stages(int mf, int ntw, int waves)
{
    const int resident = rows_resident(mf, ntw, waves);
    const int fit = (int)(160u / resident * 1024u / rows_stage_bytes(mf, ntw, waves));
    return resident == 2 && fit > 4 ? 4 : fit;
}
constexpr uint32_t rows_lds_bytes(int mf, int ntw, int waves)
{
    return (uint32_t)rows_stages(mf, ntw, waves) * rows_stage_bytes(mf, ntw, waves);
}

// A block = 16 * MF rows of x by W * NTW tiles of one of the call's weights; a unit = one
// 128-column step of a block.  The units of all blocks form one line, block after block, and
// workgroup g takes the units [g U, (g + 1) U) of it, whichever blocks they belong to: every
// compute unit gets the same number of steps for any shape (gate|up at 67 rows: 136 blocks of
// 40 steps on 256 compute units are 21.25 steps each; whole blocks would keep 120 of them idle,
// thirds of blocks would run in two rounds).  A block that one workgroup finishes alone is stored as
// output; the workgroups that share a block leave partial sums, which a second kernel adds in
// their order.
// Everything a unit needs - the rows of x, shared by the waves, and each wave's own codes and
// metadata - is written to LDS by LDS-direct loads, so the units in flight (two to four ahead of
// the arithmetic, across the end of a block) cost no registers and one counted wait per unit covers
// all of them: the loads are asm statements in one in-order queue that the compiler adds nothing
// to.  Two waves share a SIMD and overlap one's dequantization with the other's matrix
// instructions.  The weight is rounded as in the other GEMM kernels, w16 = fp16(s*q + b), and
// multiplied with the weights as the first operand: lane (r, kq) holds row 16*i + r, columns
// tile*16 + 4*kq .. + 3.
template <int MF, int NTW, int W>
__global__ void __launch_bounds__(64 * W, 2) q4_rows_kernel(const GemmGroup group)
{
    extern __shared__ uint4 rows_lds[];
    constexpr int TPB = W * NTW;
    constexpr int R = rows_stages(MF, NTW, W);
    constexpr int XJ = (4 * MF + W - 1) / W;  // loads of x per wave and unit, four rows each
    constexpr int S = XJ + NTW + 1;           // loads a wave puts in flight per unit
    static_assert(NTW <= 2, "a wave's metadata records are one load");
    static_assert(R >= 3 && S * (R - 1) <= 63, "two units ahead at least; the load counter has six bits");
    constexpr uint32_t STAGE = rows_stage_bytes(MF, NTW, W), CODES = MF * 4096u, METAS = CODES + TPB * 1024u;
    typedef __attribute__((address_space(3))) void *lds_ptr;

    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r = lane & 15u, kq = lane >> 4;
    const GemmParams &shared = group.shared;
    const uint32_t M = shared.M, K = shared.K, T = shared.T, U = shared.units, wrap_steps = shared.wrap_steps;
    const _Float16 *const x = shared.x;
    const uint32_t first_unit = blockIdx.x * U;
    const uint32_t count = first_unit + U < shared.total_units ? U : shared.total_units - first_unit;  // never 0

    // Lane offsets into x, fixed for the whole kernel.  Rows beyond M re-read the last row; a load
    // beyond the block's rows (4 MF loads do not always divide by the waves) repeats the last one.
    uint32_t x_lane[XJ], x_row[XJ];
#pragma unroll
    for (int j = 0; j < XJ; ++j) {
        const uint32_t load = XJ * wave + j;
        x_row[j] = 4u * (load < 4u * MF ? load : 4u * MF - 1u);
        const uint32_t local = x_row[j] + kq, m = local < M ? local : M - 1u;
        x_lane[j] = (m * K + 8u * (r ^ (local & 15u))) * (uint32_t)sizeof(_Float16);
    }
    // when K is an odd multiple of 64 the upper half of the last step does not exist (its codes and
    // metadata are zero): such lanes read the lower half again, 64 columns back in their row
    const bool odd_tail = K % kStepColumns != 0u;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr)rows_lds);

    // The unit fetched next: its step, and where its block's records lie.  Tiles beyond the matrix
    // re-read the last tile's codes and the last metadata word: in bounds, and never stored.
    uint32_t fetch_block = first_unit / T, fetch_step = first_unit % T, fetched = 0;
    const char *fetch_codes = nullptr, *fetch_meta = nullptr;
    uint32_t fetch_NT = 0, fetch_tile[NTW], meta_lane = 0;
    auto enter_block = [&]() {
        uint32_t t = 0;
#pragma unroll
        for (uint32_t i = 1; i < kMaxTargets; ++i)
            if (i < group.shared.targets && fetch_block >= group.target[i].first_block) t = i;
        fetch_codes = (const char *)group.target[t].codes;
        fetch_meta = (const char *)group.target[t].meta;
        fetch_NT = group.target[t].NT;
        const uint32_t tile0 = (fetch_block - group.target[t].first_block) * TPB + wave * NTW;
#pragma unroll
        for (int tile = 0; tile < NTW; ++tile) fetch_tile[tile] = tile0 + tile < fetch_NT ? tile0 + tile : fetch_NT - 1u;
        const uint32_t at = tile0 * 128u + lane * 4u, last = fetch_NT * 128u - 4u;
        meta_lane = at < last ? at : last;
    };
    auto fetch = [&](uint32_t slot) {
        const uint32_t x_step = fetch_step >= wrap_steps ? fetch_step - wrap_steps : fetch_step;
        const char *const x_at = uniform((const char *)(x + (size_t)x_step * kStepColumns));
        const uint32_t at = __builtin_amdgcn_readfirstlane(lds0 + slot * STAGE);
        const bool tail = odd_tail && fetch_step + 1u == T;
#pragma unroll
        for (int j = 0; j < XJ; ++j) {
            const uint32_t octet = r ^ ((x_row[j] + kq) & 15u);
            load_lds_x4<false>(tail && octet >= 8u ? x_lane[j] - 128u : x_lane[j], x_at, __builtin_amdgcn_readfirstlane(at + x_row[j] * 256u));
        }
        const size_t record = (size_t)fetch_step * fetch_NT;
#pragma unroll
        for (int t = 0; t < NTW; ++t)
            load_lds_x4<true>(lane * 16u, uniform(fetch_codes + (record + fetch_tile[t]) * 1024u), at + CODES + (wave * NTW + t) * 1024u);
        load_lds_x1(meta_lane, uniform(fetch_meta + record * 128u), at + METAS + wave * 256u);
        fetched += 1u;
        if (++fetch_step == T) {
            fetch_step = 0;
            fetch_block += 1u;
            if (fetched < count) enter_block();
        }
    };

    floatx4 acc[NTW][MF];
    auto clear = [&]() {
#pragma unroll
        for (int t = 0; t < NTW; ++t)
#pragma unroll
            for (int i = 0; i < MF; ++i) acc[t][i] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    };
    clear();
    const NibbleMasks masks = nibble_masks();
    uint32_t block = fetch_block, step = fetch_step;  // of the unit worked on
    uint32_t begin = step;                            // the first step of the block that this workgroup takes

    enter_block();
    static_for<R - 1>([&](auto i_c) {
        if ((uint32_t) decltype(i_c)::value < count) fetch(decltype(i_c)::value);
    });
    uint32_t slot = 0;
    for (uint32_t i = 0; i < count; ++i) {
        // this wave's loads of unit i have landed once only those of the younger units are left
        const uint32_t younger = count - 1u - i;
        if (younger >= (uint32_t)(R - 2)) {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(S * (R - 2)) : "memory");
        } else {
            static_for<R - 2>([&](auto n_c) {
                if (younger == (uint32_t) decltype(n_c)::value)
                    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(S * decltype(n_c)::value) : "memory");
            });
        }
        // behind the barrier every wave's have, and every wave has read the last of unit i - 1,
        // whose slot the fetch of unit i + R - 1 fills
        asm volatile("s_barrier" ::: "memory");
        if (fetched < count) fetch(slot == 0u ? R - 1u : slot - 1u);

        const char *const stage = (const char *)rows_lds + slot * STAGE;
        uint4 codes[NTW];
        uint2 meta[NTW];
#pragma unroll
        for (int t = 0; t < NTW; ++t) {
            codes[t] = *(const uint4 *)(stage + CODES + (wave * NTW + t) * 1024u + lane * 16u);
            meta[t] = *(const uint2 *)(stage + METAS + wave * 256u + t * 128u + r * 8u);
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
        if (++step < T && i + 1u < count) continue;

        // ---- the last unit of this block here: outputs, or partial sums
        const bool partial = begin != 0u || step != T;
        uint32_t local = block;
        const GemmParams p = select_target(group, local);
        const uint32_t sharer = blockIdx.x - block * T / U;  // number among the workgroups that share the block
        // The two common cases - 16-byte pieces of partial sums, fp16 outputs that need nothing done
        // to them - as straight code; everything else one fragment after the other
        // through one copy of it (straight code for every fragment was 2700 to 10600 lines of
        // assembly, more than the instruction cache holds; one copy for the common cases too made
        // the 27B down projection at 67 rows 40 instead of 33 us).
        const bool plain = !p.pair && p.row_scale == nullptr && p.residual == nullptr && p.y_dtype == MI355Q_F16;
        if (partial || plain) {
            const uint32_t columns = padded_columns(p.N);
            float *const sums = p.partials + (size_t)sharer * M * columns;
#pragma unroll
            for (int t = 0; t < NTW; ++t) {
                const uint32_t n = (local * TPB + wave * NTW + t) * kTileRows + 4u * kq;
#pragma unroll
                for (int f = 0; f < MF; ++f) {
                    const uint32_t m = 16u * f + r;
                    if (m >= M || n >= p.N) continue;
                    const size_t at = (size_t)m * p.N + n;
                    if (partial) {
                        *(floatx4 *)(sums + (size_t)m * columns + n) = acc[t][f];
                    } else if (!p.wide_stores) {
#pragma unroll
                        for (uint32_t j = 0; j < 4u; ++j)
                            if (n + j < p.N) ((_Float16 *)p.y)[at + j] = (_Float16)acc[t][f][j];
                    } else {
                        typedef _Float16 half4v __attribute__((ext_vector_type(4)));
                        const floatx4 v = acc[t][f];
                        *(half4v *)((_Float16 *)p.y + at) = half4v{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
                    }
                }
            }
        } else
#pragma nounroll
        for (uint32_t e = 0; e < (uint32_t)(NTW * MF); ++e) {
            floatx4 values = acc[0][0];
            static_for<NTW * MF>([&](auto e_c) {
                constexpr int at = decltype(e_c)::value;
                if (e == (uint32_t)at) values = acc[at / MF][at % MF];
            });
            const uint32_t n = (local * TPB + wave * NTW + e / MF) * kTileRows + 4u * kq;
            uint32_t m = 16u * (e % MF) + r;
            bool stored = m < M && n < p.N;
            if (p.pair) {  // rows 2m and 2m + 1 are adjacent lanes
#pragma unroll
                for (int j = 0; j < 4; ++j) values[j] += __shfl_xor(values[j], 1, 64);
                stored = stored && (m & 1u) == 0u;
                m >>= 1;
            }
            if (stored) finish_four(p, m, n, values);
        }
        // the stores are in the same queue as the fetches under way: with both gone the counts
        // above are fetches again (a builtin, so that the compiler, too, knows that its own loads
        // and stores are done and adds no wait to the loop)
        __builtin_amdgcn_s_waitcnt(0x0f70);
        clear();
        block += 1u;
        step = begin = 0;
    }
}

}  // namespace mi355q
