// Device code of the affine-Q4 linear for 17..128 rows of x: more rows than the streaming kernel
// takes, too few to keep the matrix cores busy; and for 65..256 rows of fp32 activations by weights of short rows.
// Bound by the multiplying waves' own chain of reads from LDS, dequantization and matrix instructions, one wave a SIMD (us,
// two of 17408 x 5120 at 32 and 67 rows 32.2 and 44.4; without any load 32.2 and 44.2, without arithmetic 27.4 and
// 38.3; with eight multiplying waves instead of four it took 5 % longer at 32 rows, 9 % at 48), by power (on another GPU 35.9 and 49.6;
// with zeros in x 33.7 and 44.3, in x and the codes 32.0 and 41.5), and by what a launch costs besides (the second
// kernel behind shared blocks 4 to 6 us).
#pragma once
#include "q4_gemm_device.h"

namespace mi355q {

// A block = 16 * MF fp16 rows of x by 4 * NT / KS tiles of one of the call's weights; a unit = one
// 128-column step of a block.  Eight waves, two on a SIMD: four that only fetch, everything by LDS-direct
// loads, and four that only multiply.  A wave that issues a load is held until the load has been
// taken, and with both in every wave a unit took the sum of the two (80 rows x 256 columns: 0.77 us for the loads,
// 1.07 for the arithmetic, 1.75 together; without any wait for the data 1.68).
// The multiplying waves share a unit as KS parts of its columns by 4 / KS groups of NT tiles.  With KS = 2 its rows are
// read from LDS twice instead of four times, and two waves exchange halves of their sums when the block is done, at the
// workgroup's barriers (a wait for the other wave alone, by polling a word in LDS: layers of 17 to 48 rows 0.9 % more time, of
// 49 to 96 rows 1 to 1.6 %).
template <int MF, int NT, int KS, bool PAIR>
struct RowsShape {
    static constexpr int kTiles = 4 / KS * NT, kQuarters = 4 / KS;
    static constexpr int kFragments = PAIR ? MF / 2 : MF;  // of outputs
    // One unit in LDS, a load brings 1 KiB: four rows of x; a tile's codes, eight tiles' metadata.  The rows, which
    // come from the L2, and the codes, which come from HBM, have rings and waves of their own.
    static constexpr int kRowLoads = 4 * MF, kCodeLoads = kTiles + (kTiles + 7) / 8;
    // KiB: four fragments of sums from each multiplying wave, two where the rings leave no more
    static constexpr int kExchange = KS == 1 ? 0 : 3 * kRowLoads + 3 * kCodeLoads + 16 <= 160 ? 16 : 8;
    static constexpr int kRowSlots = 4 * kRowLoads + 4 * kCodeLoads + kExchange <= 160 ? 4 : 3;
    // Four units of codes: with up to six, requests to HBM run further ahead of the multiplying waves than they are of use
    // (us, six and four units: two of 17408 x 5120 at 32 rows 32.7 and 31.5, at 67 rows 45 and 43.7; 5120 x 17408 at 67
    // rows 28.2 and 27.4), and three are too few (6144 + 1024 + 1024 x 5120 at 48 rows 15.4 and, three, 19.8).
    static constexpr int kCodeFit = (160 - kExchange - kRowSlots * kRowLoads) / kCodeLoads, kCodeSlots = kCodeFit > 4 ? 4 : kCodeFit;
    static constexpr int kRounds = KS == 1 ? 0 : (NT / 2 * kFragments + kExchange / 4 - 1) / (kExchange / 4);  // of the exchange
    static constexpr int kRowWaves = 2 * kRowLoads > 5 * kCodeLoads ? 3 : 2 * kCodeLoads > 3 * kRowLoads ? 1 : 2;
    static constexpr uint32_t kRowBytes = kRowLoads * 1024u, kCodeBytes = kCodeLoads * 1024u, kCodesAt = kRowSlots * kRowBytes;
    static constexpr uint32_t kExchangeAt = kCodesAt + kCodeSlots * kCodeBytes, kLds = kExchangeAt + kExchange * 1024u;
    static_assert(!PAIR || MF % 2 == 0, "value and remainder rows in fragments of their own");
    static_assert(kRowSlots >= 3 && kCodeSlots >= 3, "a unit ahead of the one that is read ahead, at least");
};

// The units of all blocks form one line, block after block, and workgroup g takes the units
// [g U, (g + 1) U) of it, whichever blocks they belong to: every compute unit gets the same number
// of steps for any shape (gate|up at 67 rows: 136 blocks of 40 steps on 256 compute units are 21.25
// steps each; whole blocks would keep 120 of them idle, thirds of blocks would run in two rounds).
// A block that one workgroup finishes alone is stored as output; the workgroups that share a block
// leave partial sums, which a second kernel adds in their order.  The workgroups of one XCD are neighbours on the line.
// More rows than a block has make several blocks of a group of tiles, numbered next to each other, and U a multiple of a
// block's steps.
// The fetching waves run ahead, across the ends of blocks: their loads are asm statements, each wave's in one in-order
// queue of which a counted wait takes the oldest unit.  At barrier i the units up to i + 1 have landed and unit i - 1
// has been read: the multiplying waves read their operands a quarter of a unit ahead, the next unit's first ones
// before its barrier.
// The weight is rounded as in the other GEMM kernels, w16 = fp16(s*q + b), and multiplied with the weights
// as the first operand: lane (r, kq) holds row 16*i + r, columns tile*16 + 4*kq .. + 3.
// Quarter d of a step: columns 32 j + 8 d .. + 7 for j = 0..3, which in a tile's record are the 256
// adjacent bytes 16 (16 d + r) + 4 j: lane (r, j) reads one word of codes and the word of metadata of its group
// j / 2.
// PAIR: x is 2 M rows, value and rounding remainder of each of the M rows (of fp32 activations);
// a block's value rows lie in the first half of its stage, their remainders in the second.  Each has accumulators of its
// own, which are added when the block is done: in one accumulator a row's products were rounded twice as often (relative
// error against 64 bits of 2.4 to 3.0e-7 where it is 1.7 to 2.1e-7 now, K of 1216 to 2112; 0.7 % of a call's time).
template <int MF, int NT, int KS, bool PAIR>
__global__ void __launch_bounds__(512, 2) q4_rows_kernel(const GemmGroup group)
{
    extern __shared__ uint4 rows_lds[];
    typedef RowsShape<MF, NT, KS, PAIR> S;
    constexpr int TPB = S::kTiles, OF = S::kFragments, OUT_ROWS = 16 * OF;
    typedef __attribute__((address_space(3))) void *lds_ptr;

    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r = lane & 15u, kq = lane >> 4;
    const GemmParams &shared = group.shared;
    const uint32_t M = shared.M, K = shared.K, T = shared.T, U = shared.units;
    const uint32_t m_blocks = PAIR ? shared.m_blocks : 1u;  // of rows; up to 128 rows of other activations are one
    const uint32_t number = __builtin_amdgcn_readfirstlane(number_by_xcd(blockIdx.x, gridDim.x));
    const uint32_t first_unit = number * U;
    const uint32_t count = first_unit + U < shared.total_units ? U : shared.total_units - first_unit;  // never 0

    // every argument that the first loads need is asked for at once: one after the other they came in four round trips, at
    // the start of every launch
    uint32_t first_of[kMaxTargets], NT_of[kMaxTargets];
    const char *codes_of[kMaxTargets], *meta_of[kMaxTargets];
#pragma unroll
    for (uint32_t t = 0; t < kMaxTargets; ++t) {
        first_of[t] = group.target[t].first_block;
        NT_of[t] = group.target[t].NT;
        codes_of[t] = (const char *)group.target[t].codes;
        meta_of[t] = (const char *)group.target[t].meta;
        asm volatile("" ::"s"(first_of[t]), "s"(NT_of[t]), "s"(codes_of[t]), "s"(meta_of[t]));
    }
    asm volatile("" ::"s"(M), "s"(K), "s"(T), "s"(U), "s"(m_blocks), "s"(shared.total_units), "s"(shared.targets), "s"(shared.wrap_steps), "s"(shared.x));

    if (wave >= 4u) {
        // ---- A fetching wave.  Pointers run on by a step, and only at the end of a `run` of units (a block, the half step
        // at its end, the point where the rows start over) are they made anew.  Rows beyond M re-read the last row,
        // tiles beyond the matrix the last tile's codes and the last metadata, and a wave that has a piece less than the
        // others the last piece: in bounds, and never stored.
        uint32_t block = first_unit / T, step = first_unit % T, fetched = 0, run = 0;  // of the next unit
        // SLOTS of BYTES each from `ring` on; refresh() makes the pointers of unit (block, step) and its run, fetch(to) puts
        // LOADS loads of it in flight, advance() goes a step on.
        auto stream = [&](auto loads_c, auto slots_c, uint32_t ring, uint32_t bytes, auto refresh, auto fetch, auto advance)
                          __attribute__((always_inline)) {
            constexpr int LOADS = decltype(loads_c)::value, SLOTS = decltype(slots_c)::value;
            static_assert(LOADS * (SLOTS - 1) <= 63, "the load counter has six bits");
            auto next = [&](uint32_t to) __attribute__((always_inline)) {
                fetch(__builtin_amdgcn_readfirstlane(to));
                fetched += 1u;
                step += 1u;
                if (--run != 0u) {
                    advance();
                } else if (fetched < count) {
                    if (step == T) {
                        step = 0;
                        block += 1u;
                    }
                    refresh();
                }
            };
            uint32_t left = T - step < count ? T - step : count;  // units of the block worked on that are left
            refresh();
            uint32_t slot = 0;
            for (; slot < (uint32_t)(SLOTS - 1) && fetched < count; ++slot) next(ring + slot * bytes);
            slot = (SLOTS - 1) * bytes;
            // unit u has landed once only the loads of the units behind it are left
            auto landed = [&](uint32_t u) __attribute__((always_inline)) {
                const uint32_t behind = fetched > u ? fetched - 1u - u : 0u;
                static_for<SLOTS - 1>([&](auto n_c) {
                    constexpr int n = decltype(n_c)::value;
                    if (n + 2 == SLOTS ? behind >= (uint32_t)n : behind == (uint32_t)n)
                        asm volatile("s_waitcnt vmcnt(%0)" : : "n"(LOADS * n) : "memory");
                });
            };
            landed(0);
            asm volatile("s_barrier" ::: "memory");
            for (uint32_t i = 0; i < count; ++i) {
                landed(i + 1u);
                asm volatile("s_barrier" ::: "memory");
                if (fetched < count) next(ring + slot);
                slot = slot == (SLOTS - 1) * bytes ? 0u : slot + bytes;
                if constexpr (KS == 2) {
                    if (--left != 0u) continue;
                    for (int j = 0; j < 2 * S::kRounds; ++j) asm volatile("s_barrier" ::: "memory");
                    left = T < count - 1u - i ? T : count - 1u - i;
                }
            }
        };
        const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr)rows_lds);
        if (wave < 4u + S::kRowWaves) {
            constexpr int LOADS = (S::kRowLoads + S::kRowWaves - 1) / S::kRowWaves;
            const uint32_t wrap_steps = shared.wrap_steps;
            // when K is an odd multiple of 64 the upper half of the last step does not exist (its codes and
            // metadata are zero): such lanes read the lower half again, 64 columns back in their row
            const bool odd_tail = K % kStepColumns != 0u;
            uint32_t from[LOADS], at[LOADS];
#pragma unroll
            for (int j = 0; j < LOADS; ++j) {
                const uint32_t load = j * S::kRowWaves + (wave - 4u);
                at[j] = __builtin_amdgcn_readfirstlane((load < (uint32_t)S::kRowLoads ? load : S::kRowLoads - 1u) * 1024u);
            }
            const char *rows = nullptr;
            stream(
                std::integral_constant<int, LOADS>(), std::integral_constant<int, S::kRowSlots>(), lds0, S::kRowBytes,
                [&]() __attribute__((always_inline)) {
                    const uint32_t x_step = step >= wrap_steps ? step - wrap_steps : step;
                    const bool tail = odd_tail && step + 1u == T;
                    uint32_t m0 = 0;
                    if (m_blocks > 1u) {
                        uint32_t first = first_of[0];
#pragma unroll
                        for (uint32_t t = 1; t < kMaxTargets; ++t)
                            if (t < shared.targets && block >= first_of[t]) first = first_of[t];
                        m0 = (block - first) % m_blocks * OUT_ROWS;
                    }
                    rows = (const char *)(shared.x + (size_t)(PAIR ? 2u * m0 : m0) * K + (size_t)x_step * kStepColumns);
#pragma unroll
                    for (int j = 0; j < LOADS; ++j) {
                        const uint32_t row = at[j] / 256u + kq, octet = r ^ (row & 15u);  // of the stage
                        uint32_t m = PAIR ? row % OUT_ROWS : row;
                        m = m0 + m < M ? m : M - 1u - m0;
                        from[j] = ((PAIR ? 2u * m + row / OUT_ROWS : m) * K + 8u * octet) * (uint32_t)sizeof(_Float16) -
                                  (tail && octet >= 8u ? 128u : 0u);
                    }
                    run = T - step;
                    if (odd_tail && run > 1u) run -= 1u;
                    if (step < wrap_steps && wrap_steps - step < run) run = wrap_steps - step;
                },
                [&](uint32_t to) __attribute__((always_inline)) {
                    const char *const base = uniform(rows);
#pragma unroll
                    for (int j = 0; j < LOADS; ++j) load_lds_x4<false>(from[j], base, to + at[j]);
                },
                [&]() __attribute__((always_inline)) { rows += kStepColumns * sizeof(_Float16); });
        } else {
            constexpr int WAVES = 4 - S::kRowWaves, LOADS = (S::kCodeLoads + WAVES - 1) / WAVES;
            uint32_t from[LOADS], at[LOADS], stride = 0;
#pragma unroll
            for (int j = 0; j < LOADS; ++j) {
                const uint32_t load = j * WAVES + (wave - 4u - S::kRowWaves);
                at[j] = __builtin_amdgcn_readfirstlane((load < (uint32_t)S::kCodeLoads ? load : S::kCodeLoads - 1u) * 1024u);
            }
            const char *codes = nullptr, *metas = nullptr;
            stream(
                std::integral_constant<int, LOADS>(), std::integral_constant<int, S::kCodeSlots>(), lds0 + S::kCodesAt, S::kCodeBytes,
                [&]() __attribute__((always_inline)) {
                    uint32_t first = first_of[0], all = NT_of[0];
                    codes = codes_of[0];
                    metas = meta_of[0];
#pragma unroll
                    for (uint32_t t = 1; t < kMaxTargets; ++t)
                        if (t < shared.targets && block >= first_of[t]) {
                            first = first_of[t];
                            all = NT_of[t];
                            codes = codes_of[t];
                            metas = meta_of[t];
                        }
                    const uint32_t tile0 = (m_blocks > 1u ? (block - first) / m_blocks : block - first) * TPB;
                    stride = all * 1024u;
                    codes += (size_t)step * stride;
                    metas += (size_t)step * (stride / 8u);
#pragma unroll
                    for (int j = 0; j < LOADS; ++j) {
                        const uint32_t load = at[j] / 1024u, tile = tile0 + load;
                        const uint32_t meta = (tile0 + 8u * (load - TPB)) * 128u + lane * 16u, last = all * 128u - 16u;
                        from[j] = load < (uint32_t)TPB ? (tile < all ? tile : all - 1u) * 1024u + lane * 16u : meta < last ? meta : last;
                    }
                    run = T - step;
                },
                [&](uint32_t to) __attribute__((always_inline)) {
                    const char *const codes_at = uniform(codes), *const metas_at = uniform(metas);
                    static_for<LOADS>([&](auto j_c) {
                        constexpr int j = decltype(j_c)::value;
                        if (j * WAVES + WAVES <= TPB || at[j] < TPB * 1024u)
                            load_lds_x4<true>(from[j], codes_at, to + at[j]);
                        else
                            load_lds_x4<false>(from[j], metas_at, to + at[j]);
                    });
                },
                [&]() __attribute__((always_inline)) {
                    codes += stride;
                    metas += stride / 8u;
                });
        }
        return;
    }

    // ---- a multiplying wave
    floatx4 acc[NT][MF];
    auto clear = [&]() {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < MF; ++i) acc[t][i] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    };
    clear();
    const NibbleMasks masks = nibble_masks();
    uint32_t block = first_unit / T, step = first_unit % T;  // of the unit worked on
    uint32_t begin = step;                                   // the first step of the block that this workgroup takes
    uint32_t left = T - step < count ? T - step : count;     // units of this block here that are left

    // with KS = 2 a wave's tiles begin with those whose sums it keeps, the partner's
    const uint32_t part = KS == 1 ? 0u : wave % 2u, group0 = wave / KS * NT, first_quarter = part * S::kQuarters;
    constexpr int KEPT = NT / KS;
    auto tile_at = [&](int t) { return t < KEPT ? part * KEPT + t : (1u - part) * KEPT + (t - KEPT); };  // of the group
    const uint32_t rows_at = r * 256u + ((4u * kq + first_quarter) ^ r) * 16u;
    const uint32_t codes_at = S::kCodesAt + group0 * 1024u + (first_quarter * 16u + r) * 16u + kq * 4u;
    const uint32_t metas_at = S::kCodesAt + TPB * 1024u + group0 * 128u + r * 8u + kq / 2u * 4u;
    // this lane's operands: quarter d of its part is 16 d further in the rows, by their swizzle
    uint32_t row_slot = 0, code_slot = 0;  // bytes
    half8 x_frag[2][MF];
    uint32_t codes[2][NT], meta[NT];
    auto read_rows = [&](auto d_c) __attribute__((always_inline)) {
        constexpr uint32_t d = decltype(d_c)::value;
        const char *const at = (const char *)rows_lds + row_slot + (rows_at ^ (d * 16u));
#pragma unroll
        for (int m = 0; m < MF; ++m) x_frag[d % 2u][m] = __builtin_bit_cast(half8, *(const uint4 *)(at + m * 4096u));
    };
    auto read_codes = [&](auto d_c) __attribute__((always_inline)) {
        constexpr uint32_t d = decltype(d_c)::value;
        const char *const at = (const char *)rows_lds + code_slot + codes_at + d * 256u;
#pragma unroll
        for (int t = 0; t < NT; ++t) codes[d % 2u][t] = *(const uint32_t *)(at + tile_at(t) * 1024u);
    };
    auto read_meta = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; ++t) meta[t] = *(const uint32_t *)((const char *)rows_lds + code_slot + metas_at + tile_at(t) * 128u);
    };
    auto weights = [&](uint32_t word, uint32_t of) __attribute__((always_inline)) {
        half8 scale, bias;
        meta_to_half(of, scale, bias);
        return dequant8(word, masks, scale, bias);
    };
    // the block's outputs: their arguments, too, are there before they are needed
    uint32_t local;
    GemmParams p;
    auto enter_block = [&]() __attribute__((always_inline)) {
        local = block;
        p = select_target(group, local);
        asm volatile("" ::"s"(p.y), "s"(p.residual), "s"(p.partials), "s"(p.row_scale), "s"(p.N), "s"(p.wide_stores), "s"(p.y_dtype),
                     "s"(p.residual_dtype), "s"(p.residual_is_bias));
    };
    enter_block();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    read_meta();
    read_codes(std::integral_constant<int, 0>());
    read_rows(std::integral_constant<int, 0>());
    half8 w16 = weights(codes[0][0], meta[0]);
    for (uint32_t behind = count - 1u;; --behind) {  // units behind this one
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        left -= 1u;
        step += 1u;
        // A tile's weights are made while the matrix instructions of the tile before it run.
        static_for<S::kQuarters * NT>([&](auto turn_c) __attribute__((always_inline)) {
            constexpr int turn = decltype(turn_c)::value, d = turn / NT, t = turn % NT;
            constexpr auto d_next = std::integral_constant<int, (d + 1) % S::kQuarters>();
            if constexpr (t == 0) {
                if constexpr (d + 1 == S::kQuarters) {
                    row_slot = row_slot == (S::kRowSlots - 1) * S::kRowBytes ? 0u : row_slot + S::kRowBytes;
                    code_slot = code_slot == (S::kCodeSlots - 1) * S::kCodeBytes ? 0u : code_slot + S::kCodeBytes;
                }
                read_codes(d_next);
                read_rows(d_next);
            }
            half8 next;
            if constexpr (turn + 1 == S::kQuarters * NT) {
                read_meta();
                next = weights(codes[0][0], meta[0]);
            } else {
                next = weights(codes[(turn + 1) / NT % 2][(turn + 1) % NT], meta[(turn + 1) % NT]);
            }
#pragma unroll
            for (int m = 0; m < MF; ++m)
                acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w16, x_frag[d % 2][m], acc[t][m], 0, 0, 0);
            w16 = next;
            // the weights' vector instructions between the matrix instructions: a wave issues in order, and one of those
            // waits for the one before it
#pragma unroll
            for (int m = 0; m < (MF * NT < 32 ? MF : 0); ++m) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, (14 + MF - 1) / MF, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        if (left != 0u) continue;

        // ---- the last unit of this block here: outputs, or partial sums
        if constexpr (PAIR) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int f = 0; f < OF; ++f)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[t][f][j] += acc[t][f + OF][j];
        }
        if constexpr (KS == 2) {
            constexpr int AT_ONCE = S::kExchange / 4;
            char *const mine = (char *)rows_lds + S::kExchangeAt + wave * (AT_ONCE * 1024u) + lane * 16u;
            const char *const theirs = (const char *)rows_lds + S::kExchangeAt + (wave ^ 1u) * (AT_ONCE * 1024u) + lane * 16u;
            static_for<S::kRounds>([&](auto round_c) __attribute__((always_inline)) {
                constexpr int from = AT_ONCE * decltype(round_c)::value, until = from + AT_ONCE < KEPT * OF ? from + AT_ONCE : KEPT * OF;
                asm volatile("s_barrier" ::: "memory");  // the round before has been read
#pragma unroll
                for (int e = from; e < until; ++e) *(floatx4 *)(mine + (e - from) * 1024) = acc[KEPT + e / OF][e % OF];
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
                for (int e = from; e < until; ++e) {
                    const floatx4 more = *(const floatx4 *)(theirs + (e - from) * 1024);
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[e / OF][e % OF][j] += more[j];
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            });
        }
        const bool partial = begin != 0u || step != T;
        const uint32_t sharer = number - block * T / U;  // number among the workgroups that share the block
        uint32_t m0 = 0, block_n = local;
        if (m_blocks > 1u) {
            m0 = __builtin_amdgcn_readfirstlane(local % m_blocks * OUT_ROWS);
            block_n = local / m_blocks;
        }
        // unknown to the compiler, which would else keep every row's address in registers all the time
        asm volatile("" : "+s"(m0));
        const uint32_t n0 = (block_n * TPB + group0 + part * KEPT) * kTileRows + 4u * kq;
        // The common cases - 16-byte pieces of partial sums, fp16 outputs that need nothing done to them, fp32
        // outputs - as straight code; everything else one fragment after the other
        // through one copy of it (straight code for every fragment was 2700 to 10600 lines of
        // assembly, more than the instruction cache holds; one copy for the common cases too made
        // the 27B down projection at 67 rows 40 instead of 33 us).
        const bool plain = p.row_scale == nullptr && p.residual == nullptr && p.y_dtype == MI355Q_F16;
        if (partial || plain) {
            const uint32_t columns = padded_columns(p.N);
            float *const sums = p.partials + (size_t)sharer * M * columns;
#pragma unroll
            for (int t = 0; t < KEPT; ++t) {
                const uint32_t n = n0 + t * kTileRows;
#pragma unroll
                for (int f = 0; f < OF; ++f) {
                    const uint32_t m = m0 + 16u * f + r;
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
        } else if (p.y_dtype == MI355Q_F32 && (p.residual == nullptr || p.residual_dtype == MI355Q_F32) &&
                   (PAIR || (p.wide_stores && (uintptr_t)p.residual % 16u == 0u))) {
            // The loads of a tile's residuals are on their way together.  Outputs without 16-byte pieces here, too, but of pairs
            // only: with this code in the other forms the loop above came out 6 to 8 % slower (two of 13440 x 3840 at 35 rows
            // 20.0 -> 21.9 us).
            const bool wide = !PAIR || (p.wide_stores && (uintptr_t)p.residual % 16u == 0u);
            float scale[OF];
#pragma unroll
            for (int f = 0; f < OF; ++f) {
                const uint32_t m = m0 + 16u * f + r;
                scale[f] = p.row_scale == nullptr ? 1.0f : p.row_scale[m < M ? m : M - 1u];
            }
#pragma unroll
            for (int t = 0; t < KEPT; ++t) {
                const uint32_t n = n0 + t * kTileRows;
                if (n >= p.N) continue;
                floatx4 more[OF];
#pragma unroll
                for (int f = 0; f < OF; ++f) more[f] = floatx4{-0.0f, -0.0f, -0.0f, -0.0f};  // (which adds nothing, also to -0)
                if (p.residual != nullptr) {
#pragma unroll
                    for (int f = 0; f < OF; ++f) {
                        const uint32_t m = m0 + 16u * f + r;
                        const float *const from = (const float *)p.residual + (p.residual_is_bias ? 0 : (size_t)(m < M ? m : M - 1u) * p.N);
                        if (wide) {
                            more[f] = *(const floatx4 *)(from + n);
                        } else {
#pragma unroll
                            for (uint32_t j = 0; j < 4u; ++j) more[f][j] = from[n + j < p.N ? n + j : p.N - 1u];
                        }
                    }
                }
#pragma unroll
                for (int f = 0; f < OF; ++f) {
                    const uint32_t m = m0 + 16u * f + r;
                    float *const to = (float *)p.y + (size_t)m * p.N + n;
                    floatx4 value;
#pragma unroll
                    for (int j = 0; j < 4; ++j) value[j] = acc[t][f][j] * scale[f] + more[f][j];
                    if (m >= M) continue;
                    if (wide) {
                        *(floatx4 *)to = value;
                    } else {
#pragma unroll
                        for (uint32_t j = 0; j < 4u; ++j)
                            if (n + j < p.N) to[j] = value[j];
                    }
                }
            }
        } else
#pragma nounroll
        for (uint32_t e = 0; e < (uint32_t)(KEPT * OF); ++e) {
            floatx4 values = acc[0][0];
            static_for<KEPT * OF>([&](auto e_c) {
                constexpr int at = decltype(e_c)::value;
                if (e == (uint32_t)at) values = acc[at / OF][at % OF];
            });
            const uint32_t n = n0 + e / OF * kTileRows, m = m0 + 16u * (e % OF) + r;
            if (m < M && n < p.N) finish_four(p, m, n, values);
        }
        if (behind == 0u) break;
        clear();
        block += 1u;
        step = begin = 0;
        left = T < behind ? T : behind;
        enter_block();
    }
}

// Blocks of TILES tiles (q4_rows_*.hip: one file of instantiations per number of tiles, so that they
// compile side by side): the kernel for mf fragments.
template <int NT, int KS>
static hipError_t launch_rows_of(mi355q_context *ctx, int mf, bool pair, uint32_t groups, const GemmGroup &group)
{
    auto of = [&](auto mf_c, auto pair_c) {
        constexpr int MF = decltype(mf_c)::value;
        constexpr bool PAIR = decltype(pair_c)::value;
        // whole columns to a wave: up to 32 rows of 16-bit activations by 8 and 16 tiles, whose reading from LDS is cheaper than
        // an exchange (layers of 17 to 32 rows 0.8 % less time, of 33 to 48 0.8 % more, fp32 calls of 9 to 16 as much and a
        // larger error), and 96 and 128 rows by 16 tiles, for the accumulators' sake
        constexpr int SPLIT = (NT >= 4 && MF == 2 && !PAIR) || (NT == 8 && MF >= 6) ? 2 : 1;
        typedef RowsShape<MF, NT / SPLIT, KS / SPLIT, PAIR> S;
        bool &raised = ctx->rows_lds_raised[MF - 1][PAIR][S::kTiles / 8];
        const auto kernel = q4_rows_kernel<MF, NT / SPLIT, KS / SPLIT, PAIR>;
        if (!raised) {  // per context (a context belongs to one device and serialises its calls)
            hipError_t status = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::kLds);
            if (status != hipSuccess) return status;
            raised = true;
        }
        return launch(ctx, kernel, dim3(groups), dim3(512), S::kLds, group);
    };
    if (pair) {
        switch (mf) {
        case 2: return of(std::integral_constant<int, 2>(), std::true_type());
        case 4: return of(std::integral_constant<int, 4>(), std::true_type());
        case 6: return of(std::integral_constant<int, 6>(), std::true_type());
        default: return of(std::integral_constant<int, 8>(), std::true_type());
        }
    }
    switch (mf) {
    case 2: return of(std::integral_constant<int, 2>(), std::false_type());
    case 3: return of(std::integral_constant<int, 3>(), std::false_type());
    case 4: return of(std::integral_constant<int, 4>(), std::false_type());
    case 5: return of(std::integral_constant<int, 5>(), std::false_type());
    case 6: return of(std::integral_constant<int, 6>(), std::false_type());
    default: return of(std::integral_constant<int, 8>(), std::false_type());
    }
}
hipError_t q4_rows_launch_4(mi355q_context *ctx, int mf, bool pair, uint32_t groups, const GemmGroup &group);
hipError_t q4_rows_launch_8(mi355q_context *ctx, int mf, bool pair, uint32_t groups, const GemmGroup &group);
hipError_t q4_rows_launch_16(mi355q_context *ctx, int mf, bool pair, uint32_t groups, const GemmGroup &group);

}  // namespace mi355q
