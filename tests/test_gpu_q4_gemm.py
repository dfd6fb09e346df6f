"""GPU parity of the prefill GEMM (M > 16) against the CPU oracle, through the C ABI.

The GEMM rounds each weight to fp16 before an fp16 x fp16 multiply with fp32 accumulation
(as the reference's batched kernels and its scalar check do, minimax_h3_m3_gemm.m:87-104), so
the gate compares with the oracle's fp16-weight flavour in double accumulation:
max_i |y_i - ref_i| / max(|ref_i|, 1e-2*rms(ref)) <= 1e-3.  The distance to the exact-weight
result is reported against rms(ref) (the weight rounding itself, ~2^-12 per weight)."""
import re

import numpy as np
import pytest

from conftest import bf16_bits, q4_relative_error

pytestmark = pytest.mark.gpu


def make_x(engine, seed, M, K):
    return engine.synth_normal_f32(seed, 1.0, M * K).reshape(M, K)


def run_case(engine, oracle, gpu, N, K, M, meta_kind, x_dtype, y_dtype, columns=None, seed=5,
             residual=False):
    quants, meta_a, meta_b = engine.synth_q4_affine(seed, 0.02, N, K, meta_kind)
    x32 = make_x(engine, seed + 1, M, K)
    if x_dtype == engine.F16:
        x = x32.astype(np.float16)
        x_ref, x_kind = x, oracle.X_F16
    elif x_dtype == engine.BF16:
        x = bf16_bits(x32).reshape(M, K)
        # the kernel multiplies fp16: bf16 values in fp16's normal range convert exactly
        x_ref, x_kind = x, oracle.X_BF16
    else:
        x = x32
        x_ref, x_kind = x32, oracle.X_F32  # fp32 rows go in as (value, remainder) pairs: not rounded
    res = engine.synth_normal_f32(seed + 2, 1.0, M * N).reshape(M, N) if residual else None
    weight = gpu.q4_prepare(quants, meta_a, meta_b, N, K, meta_kind)
    try:
        print(f"gemm case N={N} K={K} M={M} meta={meta_kind} x={x_dtype} y={y_dtype}", flush=True)
        y = gpu.q4_linear(weight, x, x_dtype, y_dtype, res, engine.F32)
    finally:
        weight.destroy()
    windows = columns if columns else [(0, N)]
    if isinstance(windows, tuple):
        windows = [windows]
    assert np.all(np.isfinite(np.asarray(y, dtype=np.float64)))
    if y_dtype == engine.BF16:
        y = (y.astype(np.uint32) << 16).view(np.float32)
    error = 0.0
    for lo, hi in windows:
        ref = oracle.q4_linear(quants, meta_a, meta_b, meta_kind, N, K, x_ref, x_kind, M,
                               weight_rounding=oracle.W_ROUND_F16, rows=(lo, hi))[:, lo:hi]
        exact = oracle.q4_linear(quants, meta_a, meta_b, meta_kind, N, K, x_ref, x_kind, M,
                                 rows=(lo, hi))[:, lo:hi]
        if residual:
            ref, exact = ref + res[:, lo:hi], exact + res[:, lo:hi]
        got = np.asarray(y, dtype=np.float64)[:, lo:hi]
        window_error = q4_relative_error(got, ref)
        tolerance = 2.0 ** -8 if y_dtype == engine.BF16 else 1e-3
        assert window_error <= tolerance, f"columns {lo}..{hi}: relative error {window_error:.3e}"
        rms = np.sqrt(np.mean(exact * exact))
        drift = float(np.max(np.abs(got - exact)) / rms)
        # a bf16 output adds its own rounding: half an ulp (2^-9 relative) of the largest output
        limit = 2e-3 + (2.0 ** -9 * float(np.max(np.abs(exact)) / rms) if y_dtype == engine.BF16 else 0.0)
        assert drift <= limit, f"columns {lo}..{hi}: vs exact weights {drift:.3e}"
        error = max(error, window_error)
    return error


@pytest.mark.parametrize("N,K,M", [(256, 128, 17), (512, 1024, 64), (272, 192, 130), (100, 64, 33),
                                   (1040, 2048, 257)])
@pytest.mark.parametrize("meta_kind", [0, 1])
def test_small_shapes(engine, oracle, gpu, N, K, M, meta_kind):
    run_case(engine, oracle, gpu, N, K, M, meta_kind, engine.F16, engine.F32)


def geometry_windows(N):
    """16-column windows (whole weight tiles) placed by the launch geometry of the GEMM kernels:
    a workgroup takes 16, 17 (16 + one tile shared by its four waves) or 20 consecutive tiles,
    four or five per wave.  Tiles 0, 5, 10 and 15 fall to the four waves of the first workgroup
    whichever of the three it is; tile 16 is the shared seventeenth tile of the first 17-tile
    workgroup; the others sit in an interior workgroup (its shared tile, and a tile of its last
    wave) and in the last workgroup, down to the last (possibly partly filled) tile."""
    tiles = (N + 15) // 16
    middle = tiles // 17 // 2
    picks = {0, 5, 10, 15, 16, 17 * middle + 16, 17 * middle + 13, 20 * (tiles // 20 // 2) + 19,
             16 * (tiles // 16 // 2) + 7, tiles - 20, tiles - 17, tiles - 1}
    return [(16 * t, min(16 * t + 16, N)) for t in sorted(t for t in picks if 0 <= t < tiles)]


@pytest.mark.parametrize("M", [512, 2048])
@pytest.mark.parametrize("N,K", [(17408, 5120), (5120, 17408)])
def test_prefill_shapes(engine, oracle, gpu, N, K, M):
    """Headline configuration 4 (27B MLP shapes at prefill row counts): bf16 scale/bias, fp16
    activations, fp16 output.  The oracle checks every row of x at full K on a dozen 16-column
    windows chosen from the launch geometry (see geometry_windows); the rest of the output is
    checked for finiteness and, below, against the streaming kernel."""
    run_case(engine, oracle, gpu, N, K, M, engine.META_BF16_PLANES, engine.F16, engine.F16,
             columns=geometry_windows(N))


def test_agrees_with_streaming_kernel_rows(engine, gpu):
    """Size-independent property: row m of the GEMM equals the M=1 streaming result for x[m]
    up to the fp16 weight rounding (the streaming kernel keeps the weight exact)."""
    N, K, M = 5120, 17408, 512
    quants, meta_a, meta_b = engine.synth_q4_affine(9, 0.02, N, K, engine.META_BF16_PLANES)
    x = make_x(engine, 10, M, K).astype(np.float16)
    weight = gpu.q4_prepare(quants, meta_a, meta_b, N, K, engine.META_BF16_PLANES)
    try:
        big = gpu.q4_linear(weight, x, engine.F16, engine.F32)
        for m in (0, 255, 511):
            one = gpu.q4_linear(weight, x[m:m + 1], engine.F16, engine.F32)
            rms = float(np.sqrt(np.mean(one.astype(np.float64) ** 2)))
            assert float(np.max(np.abs(big[m] - one[0]))) <= 2e-3 * rms
    finally:
        weight.destroy()


@pytest.mark.parametrize("x_dtype,y_dtype", [("F32", "F32"), ("BF16", "BF16"), ("F16", "F16")])
def test_dtypes_and_residual(engine, oracle, gpu, x_dtype, y_dtype):
    run_case(engine, oracle, gpu, 384, 512, 40, engine.META_F16_INTERLEAVED, getattr(engine, x_dtype),
             getattr(engine, y_dtype), residual=True)


@pytest.mark.parametrize("forced", [None, "0,1", "3,2", "6,1", "7,2"])
def test_activation_range(engine, oracle, gpu, force, forced):
    """Activations far from fp16's range on the matrix-instruction path (64 rows): fp32 and bf16
    rows of magnitude 1e4, 1e-3 and 1e-6 and rows with entries beyond 65504.  Rows that are not
    fp16 are scaled by a power of two per row and fp32 rows go in as (value, remainder) pairs, so
    the gate against the fp16-weight oracle on the caller's own x holds whatever the magnitude
    (the reference keeps fp32 activations at any row count: whisper_turbo_encoder.c:128-176,
    qwen38_m3_layer.m:375-393); with a residual and through a K split."""
    N, K, M = 528, 1536, 64
    if forced:
        force("q4_gemm", forced)
    quants, meta_a, meta_b = engine.synth_q4_affine(191, 0.02, N, K, engine.META_BF16_PLANES)
    x = make_x(engine, 192, M, K).copy()
    scales = np.ones(M, dtype=np.float32)
    scales[0::4], scales[1::4], scales[2::4] = 1e4, 1e-3, 1e-6
    x *= scales[:, None]
    x[3, 5], x[3, 77], x[7, 1000] = np.float32(1e5), np.float32(-2.5e5), np.float32(7e4)
    x_bf = bf16_bits(x).reshape(M, K)
    res = engine.synth_normal_f32(193, 1.0, M * N).reshape(M, N) * scales[:, None]
    weight = gpu.q4_prepare(quants, meta_a, meta_b, N, K, engine.META_BF16_PLANES)
    try:
        print(f"gemm activation range case forced={forced}", flush=True)
        y = gpu.q4_linear(weight, x, engine.F32, engine.F32, res, engine.F32)
        y_bf = gpu.q4_linear(weight, x_bf, engine.BF16, engine.F32)
    finally:
        weight.destroy()
    assert np.all(np.isfinite(y)) and np.all(np.isfinite(y_bf))
    ref = oracle.q4_linear(quants, meta_a, meta_b, engine.META_BF16_PLANES, N, K, x, oracle.X_F32, M,
                           weight_rounding=oracle.W_ROUND_F16) + res
    assert q4_relative_error(y, ref) <= 1e-3
    ref_bf = oracle.q4_linear(quants, meta_a, meta_b, engine.META_BF16_PLANES, N, K, x_bf, oracle.X_BF16, M,
                              weight_rounding=oracle.W_ROUND_F16)
    assert q4_relative_error(y_bf, ref_bf) <= 1e-3


@pytest.mark.parametrize("forced", ["0,1", "1,2", "2,1", "3,1", "3,3", "4,1", "5,2", "6,1", "6,3", "7,1", "7,2", "8,1", "8,2"])
def test_forced_decompositions(engine, oracle, gpu, forced, force):
    """Every kernel variant the host heuristic can pick (rows per block, tiles per wave, odd
    tile on the last wave), with and without K splits."""
    force("q4_gemm", forced)
    run_case(engine, oracle, gpu, 1104, 2176, 150, engine.META_BF16_PLANES, engine.F16, engine.F32)


@pytest.mark.parametrize("forced", ["6,1", "7,1", "7,2", "8,1"])
@pytest.mark.parametrize("K", [128, 256, 384, 640])
def test_pipelined_kernel_short_rows(engine, oracle, gpu, forced, K, force):
    """The pipelined kernel fetches three steps ahead and rotates its registers over three
    steps: rows of one to five 128-column steps exercise its prologue, the clamped fetches past
    the end and both remainder steps (alone and under a K split)."""
    force("q4_gemm", forced)
    run_case(engine, oracle, gpu, 560, K, 70, engine.META_BF16_PLANES, engine.F16, engine.F32)


@pytest.mark.parametrize("forced", ["6,1", "7,2", "8,1"])
@pytest.mark.parametrize("y_dtype", ["F16", "F32", "BF16"])
def test_pipelined_kernel_rows_of_odd_width(engine, oracle, gpu, forced, y_dtype, force):
    """N % 4 != 0: the pipelined kernel's four-at-once stores do not apply and every output leaves
    on its own (also the last, partly filled tile)."""
    force("q4_gemm", forced)
    run_case(engine, oracle, gpu, 1102, 384, 150, engine.META_BF16_PLANES, engine.F16,
             getattr(engine, y_dtype), residual=(y_dtype == "F32"))


@pytest.mark.parametrize("forced", ["6,1", "7,2", "8,2"])
@pytest.mark.parametrize("y_dtype,width", [("F16", 2), ("F32", 4), ("BF16", 2)])
def test_pipelined_kernel_output_alignment(engine, gpu, forced, y_dtype, width, force):
    """A device output pointer that is not 16-byte aligned takes the element-wise stores and must
    give the same bits as the aligned call."""
    force("q4_gemm", forced)
    N, K, M = 1104, 384, 150
    quants, meta_a, meta_b = engine.synth_q4_affine(21, 0.02, N, K, engine.META_BF16_PLANES)
    x = make_x(engine, 22, M, K).astype(np.float16)
    weight = gpu.q4_prepare(quants, meta_a, meta_b, N, K, engine.META_BF16_PLANES)
    x_ptr = gpu.to_device(x)
    y_ptr = gpu.alloc(M * N * width + 64)
    kind = {2: np.uint16, 4: np.uint32}[width]
    try:
        outputs = []
        for shift in (0, width):  # aligned, then one element further
            print(f"gemm alignment case forced={forced} y={y_dtype} shift={shift}", flush=True)
            calls = engine.make_calls([((weight, y_ptr + shift), x_ptr, engine.F16, M, getattr(engine, y_dtype))])
            gpu.q4_sequence(calls)
            gpu.sync()
            outputs.append(gpu.download(y_ptr + shift, (M, N), kind))
        assert np.array_equal(outputs[0], outputs[1])
        assert np.any(outputs[0] != 0)
    finally:
        gpu.free(x_ptr)
        gpu.free(y_ptr)
        weight.destroy()


@pytest.mark.parametrize("N,K,M,splits", [(17408, 5120, 512, 1), (1104, 2176, 150, 2), (560, 384, 70, 1)])
def test_hand_scheduled_loads_match_compiler_managed_loads(engine, gpu, force, N, K, M, splits):
    """The pipelined kernel issues its weight loads as asm statements and waits for them with its
    own counted s_waitcnt; a second build of the same kernel (the 17-tile shape) uses ordinary loads
    whose waits the compiler places.  Same bits, or a wait no longer covers its loads."""
    kind = engine.META_BF16_PLANES
    quants, meta_a, meta_b = engine.synth_q4_affine(61, 0.02, N, K, kind)
    x = make_x(engine, 62, M, K).astype(np.float16)
    weight = gpu.q4_prepare(quants, meta_a, meta_b, N, K, kind)
    try:
        force("q4_gemm", f"7,{splits}")
        print(f"gemm load forms N={N} K={K} M={M} splits={splits}", flush=True)
        scheduled = gpu.q4_linear(weight, x, engine.F16, engine.F32)
        force("gemm_loads", "plain")
        plain = gpu.q4_linear(weight, x, engine.F16, engine.F32)
    finally:
        weight.destroy()
    assert np.array_equal(scheduled.view(np.uint32), plain.view(np.uint32))
    assert np.any(scheduled != 0)



@pytest.mark.parametrize("N,K,M,forced", [(1104, 2176, 400, "6,2"), (1104, 2176, 150, "7,3"), (5120, 640, 300, "8,1"),
                                          (560, 384, 70, "6,1")])
def test_block_order_does_not_change_the_bits(engine, gpu, force, N, K, M, forced):
    """The pipelined kernel either takes its blocks in launch order or renumbers them so that the
    row blocks of one tile block run on one XCD (numbers of blocks that are and are not multiples
    of eight, with K splits, ragged last blocks): every block is computed exactly once either way,
    so the outputs are the same bits."""
    kind = engine.META_BF16_PLANES
    quants, meta_a, meta_b = engine.synth_q4_affine(71, 0.02, N, K, kind)
    x = make_x(engine, 72, M, K).astype(np.float16)
    weight = gpu.q4_prepare(quants, meta_a, meta_b, N, K, kind)
    try:
        force("q4_gemm", forced)
        print(f"gemm block order N={N} K={K} M={M} forced={forced}", flush=True)
        force("gemm_order", "launch")
        in_launch_order = gpu.q4_linear(weight, x, engine.F16, engine.F32)
        force("gemm_order", "xcd")
        renumbered = gpu.q4_linear(weight, x, engine.F16, engine.F32)
    finally:
        weight.destroy()
    assert np.array_equal(in_launch_order.view(np.uint32), renumbered.view(np.uint32))
    assert np.any(renumbered != 0)


@pytest.mark.parametrize("forced", ["1,1", "2,2", "4,1", "5,1", "6,1", "6,2", "7,1", "7,2", "8,1"])
@pytest.mark.parametrize("x_dtype,y_dtype,N", [("F32", "F32", 1104), ("F32", "F32", 1102), ("F32", "BF16", 1100),
                                               ("BF16", "BF16", 1104), ("BF16", "F16", 1100), ("BF16", "F32", 1101)])
def test_converted_activations_finish_in_the_kernel(engine, oracle, gpu, force, forced, x_dtype, y_dtype, N):
    """Activations that are not fp16: the matrix kernel's own epilogue (or the kernel that adds K
    splits) adds the two rows of a pair, undoes the row scale, adds the residual and converts.
    Ragged last tiles, widths that are and are not multiples of 4 and 8, a last block of rows that
    is partly filled, with and without a residual."""
    force("q4_gemm", forced)
    kind, K, M = engine.META_BF16_PLANES, 256, 75
    quants, meta_a, meta_b = engine.synth_q4_affine(77, 0.02, N, K, kind)
    x32 = make_x(engine, 78, M, K)
    x = x32 if x_dtype == "F32" else bf16_bits(x32).reshape(M, K)
    res = engine.synth_normal_f32(79, 1.0, M * N).reshape(M, N)
    product = oracle.q4_linear(quants, meta_a, meta_b, kind, N, K, x, oracle.X_F32 if x_dtype == "F32" else oracle.X_BF16,
                               M, weight_rounding=oracle.W_ROUND_F16)
    weight = gpu.q4_prepare(quants, meta_a, meta_b, N, K, kind)
    try:
        for residual in (None, res):
            print(f"gemm epilogue N={N} x={x_dtype} y={y_dtype} forced={forced} residual={residual is not None}", flush=True)
            y = gpu.q4_linear(weight, x, getattr(engine, x_dtype), getattr(engine, y_dtype), residual, engine.F32)
            y = (y.astype(np.uint32) << 16).view(np.float32) if y_dtype == "BF16" else y
            # a bf16 output is rounded by at most half a unit of its eight bits: 2^-8 of its value
            error = q4_relative_error(y, product if residual is None else product + res)
            assert error <= (2.0 ** -8 if y_dtype == "BF16" else 1e-3)
    finally:
        weight.destroy()


@pytest.mark.parametrize("x_dtype", ["F32", "BF16"])
@pytest.mark.parametrize("M", [9, 40, 150])
def test_targets_share_converted_activations(engine, gpu, x_dtype, M):
    """Weights of one call multiply activations that were converted once: the results of one call per
    weight up to the order of the fp32 sums, which at 17 to 128 matrix rows depends on the weights that
    share the call; above that, where each is multiplied by itself, the same bits."""
    K, widths = 384, (272, 1000, 100)
    x32 = make_x(engine, 81, M, K)
    x = x32 if x_dtype == "F32" else bf16_bits(x32).reshape(M, K)
    kind, x_dtype = engine.META_BF16_PLANES, getattr(engine, x_dtype)
    weights = [gpu.q4_prepare(*engine.synth_q4_affine(82 + i, 0.02, N, K, kind), N, K, kind) for i, N in enumerate(widths)]
    biases = [gpu.to_device(engine.synth_normal_f32(90 + i, 1.0, N)) for i, N in enumerate(widths)]
    x_ptr = gpu.to_device(x)
    outputs = [gpu.alloc(M * N * 4) for N in widths]
    try:
        results = []
        targets = list(zip(weights, outputs, biases))
        for groups in ([targets], [[t] for t in targets]):
            print(f"gemm targets M={M} x={x_dtype} calls={len(groups)}", flush=True)
            calls = engine.make_calls([(g, x_ptr, x_dtype, M, engine.F32, engine.F32, engine.RESIDUAL_IS_BIAS)
                                       for g in groups])
            gpu.q4_sequence(calls)
            gpu.sync()
            results.append([gpu.download(p, (M, N), np.uint32) for p, N in zip(outputs, widths)])
        for together, alone in zip(*results):
            assert np.any(alone != 0)
            close = np.abs(together.view(np.float32) - alone.view(np.float32))
            assert np.max(close) <= 2e-6 * np.max(np.abs(alone.view(np.float32)))
            if M == 150:
                assert np.array_equal(together, alone)
    finally:
        for pointer in [x_ptr] + outputs + biases:
            gpu.free(pointer)
        for weight in weights:
            weight.destroy()


@pytest.mark.parametrize("forced", ["11,1", "11,2", "12,1", "12,2", "12,3", "13,1", "13,2"])
@pytest.mark.parametrize("N,K,M", [(100, 64, 17), (272, 128, 32), (1102, 192, 33), (1104, 1024, 48), (560, 576, 63),
                                   (1001, 640, 67), (272, 2176, 80), (1104, 384, 96), (256, 1088, 97), (1102, 256, 128),
                                   (9000, 1920, 40)])
def test_rows_kernel(engine, oracle, gpu, force, forced, N, K, M):
    """17 to 128 rows by blocks of 4, 8 and 16 tiles: fragments of rows partly filled, tiles beyond
    the matrix, K an odd multiple of 64 (half of the last step does not exist), fewer steps than
    stages, workgroups that take one step, several blocks, or the end of one block and the
    beginning of the next."""
    force("q4_gemm", forced)
    run_case(engine, oracle, gpu, N, K, M, engine.META_BF16_PLANES, engine.F16, engine.F32, residual=True)
    run_case(engine, oracle, gpu, N, K, M, engine.META_F16_INTERLEAVED, engine.F16, engine.F16)


@pytest.mark.parametrize("forced", ["11,1", "11,5", "12,2", "12,5", "13,1", "13,5"])
@pytest.mark.parametrize("N,K,M", [(1104, 1280, 16), (1104, 192, 17), (272, 1280, 32), (1101, 640, 48), (2052, 640, 49), (64, 128, 64)])
def test_rows_kernel_pairs(engine, oracle, gpu, force, forced, N, K, M):
    """fp32 activations: value and remainder rows in fragments of their own, one to four fragments of
    outputs full and with one row more; fp32 outputs with residual rows (16-byte pieces, and a width that has
    none) and without."""
    force("q4_gemm", forced)
    run_case(engine, oracle, gpu, N, K, M, engine.META_BF16_PLANES, engine.F32, engine.F32, residual=True)
    run_case(engine, oracle, gpu, N, K, M, engine.META_F16_INTERLEAVED, engine.F32, engine.F32)


@pytest.mark.parametrize("forced,M,parts", [("11,1", 16, 2), ("12,1", 16, 2), ("13,1", 16, 2), ("11,1", 32, 2), ("12,1", 32, 2),
                                            ("13,1", 32, 2), ("11,1", 48, 2), ("12,1", 64, 2), ("13,1", 64, 1)])
@pytest.mark.parametrize("K", [1280, 5120])
def test_rows_kernel_pairs_precision(engine, oracle, gpu, force, forced, parts, M, K):
    """fp32 activations on whole blocks: an output is as near to 64 bits as sums of a row's K value products alone, in
    `parts` accumulators.  An addition of the matrix instruction (eight products; four of them an instruction) is off by
    0.424 * 2^-24 of the sum (rms over mantissas), and n of them into a sum that grows like a random walk by that times
    sqrt(n / 2); n additions in two halves by sqrt(n / 4).  A tenth more for the pieces of x and for the sample."""
    N, kind = 1024, engine.META_BF16_PLANES
    force("q4_gemm", forced)
    planes = engine.synth_q4_affine(221, 0.02, N, K, kind)
    x = make_x(engine, 222, M, K)
    weight = gpu.q4_prepare(*planes, N, K, kind)
    try:
        print(f"pairs precision M={M} K={K} forced={forced}", flush=True)
        y = gpu.q4_linear(weight, x, engine.F32, engine.F32).astype(np.float64)
    finally:
        weight.destroy()
    exact = oracle.q4_linear(*planes, kind, N, K, x, oracle.X_F32, M, weight_rounding=oracle.W_ROUND_F16)
    error = np.sqrt(np.sum((y - exact) ** 2) / np.sum(exact ** 2))
    bound = 1.1 * 0.424 * 2.0 ** -24 * np.sqrt(K / 8 / (2 * parts))
    print(f"relative error {error:.3e}, bound {bound:.3e}", flush=True)
    assert error <= bound


@pytest.mark.parametrize("K,widths,by_rows", [(1280, (1280, 1280, 1280), 3), (640, (2048, 516, 1002), 3),
                                              (640, (2048, 2564, 516, 2561), 2), (1152, (3072,), 1), (384, (1, 1536), 2)])
@pytest.mark.parametrize("M", [65, 129, 150, 193, 256])
def test_pairs_of_many_rows(engine, oracle, gpu, force, capfd, K, widths, by_rows, M):
    """65 to 256 fp32 rows by q4_rows_kernel: two to sixteen blocks of rows, the last with one row or full, weights it
    takes beside wider ones that it does not, which run behind them on the same converted activations.  Each output
    has the bits of its weight's own call, agrees with another kernel up to the order of the sums, and the first
    weight's with the oracle."""
    kind = engine.META_BF16_PLANES
    x = make_x(engine, 201, M, K)
    planes = [engine.synth_q4_affine(202 + i, 0.02, N, K, kind) for i, N in enumerate(widths)]
    weights = [gpu.q4_prepare(*p, N, K, kind) for p, N in zip(planes, widths)]
    biases = [gpu.to_device(engine.synth_normal_f32(210 + i, 1.0, N)) for i, N in enumerate(widths)]
    x_ptr = gpu.to_device(x)
    outputs = [gpu.alloc(M * N * 4) for N in widths]
    try:
        results, printed = [], []
        targets = list(zip(weights, outputs, biases))
        for how, groups in (("", [targets]), ("", [[t] for t in targets]), ("4,1", [[t] for t in targets])):
            print(f"pairs M={M} K={K} widths={widths} forced={how}", flush=True)
            force("q4_gemm", how)
            force("trace", "1")
            for pointer, N in zip(outputs, widths):
                gpu.upload(pointer, np.full((M, N), np.nan, np.float32))
            capfd.readouterr()
            gpu.q4_sequence(engine.make_calls([(g, x_ptr, engine.F32, M, engine.F32, engine.F32, engine.RESIDUAL_IS_BIAS)
                                               for g in groups]))
            gpu.sync()
            printed.append(capfd.readouterr().err)
            results.append([gpu.download(p, (M, N), np.float32) for p, N in zip(outputs, widths)])
        line = f"q4 rows M={M}"
        assert [p.count(line) for p in printed] == [1, by_rows, 0]
        for together, alone, other in zip(*results):
            assert np.array_equal(together, alone)
            # K products of one row, of values and of remainders, summed in another order
            assert np.max(np.abs(alone - other)) <= 2 * K * 2.0 ** -24 * np.max(np.abs(other))
        ref = oracle.q4_linear(*planes[0], kind, widths[0], K, x, oracle.X_F32, M, weight_rounding=oracle.W_ROUND_F16)
        ref = ref + gpu.download(biases[0], (1, widths[0]), np.float32)
        assert q4_relative_error(np.asarray(results[1][0], np.float64), ref) <= 1e-3
    finally:
        for pointer in [x_ptr] + outputs + biases:
            gpu.free(pointer)
        for weight in weights:
            weight.destroy()


@pytest.mark.parametrize("forced,tiles,rows,blocks", [
    ("11,1", 4, 16, 1), ("12,9", 8, 16, 3), ("13,5", 16, 16, 2), ("11,6", 4, 32, 2), ("11,11", 4, 48, 3), ("11,8", 4, 64, 2), ("12,2", 8, 32, 1), ("12,10", 8, 32, 3),
    ("12,7", 8, 48, 2), ("12,12", 8, 64, 3), ("13,2", 16, 32, 1), ("13,6", 16, 32, 2), ("13,10", 16, 32, 3)])
@pytest.mark.parametrize("y_dtype,residual_dtype,shift", [("F32", "F32", 0), ("F32", "F32", 1), ("F32", "F16", 0), ("F16", "F32", 0),
                                                          ("BF16", "BF16", 1), ("F32", None, 0)])
@pytest.mark.parametrize("K,M", [(384, 150), (1152, 257)])
def test_blocks_of_pairs(engine, gpu, force, capfd, forced, tiles, rows, blocks, y_dtype, residual_dtype, shift, K, M):
    """Every block of fp32 pairs beyond 64 rows, one to three a workgroup: runs that end inside a weight and in the next
    one, more blocks than compute units and fewer, a last block of rows partly filled, tiles beyond the matrix, widths
    with and without 16-byte pieces; residual rows of every type, outputs of every type, also one element off
    their alignment.  The bits do not depend on the block."""
    kind, widths = engine.META_BF16_PLANES, (1284, 330, 64, 1002)
    x = make_x(engine, 231, M, K)
    weights = [gpu.q4_prepare(*engine.synth_q4_affine(232 + i, 0.02, N, K, kind), N, K, kind) for i, N in enumerate(widths)]
    cell = {"F32": np.float32, "F16": np.float16, "BF16": np.uint16}

    def rows_of(seed, N, dtype):
        values = engine.synth_normal_f32(seed, 1.0, M * N).reshape(M, N)
        return bf16_bits(values) if dtype == "BF16" else values.astype(cell[dtype])

    residuals = [None if residual_dtype is None else gpu.to_device(rows_of(240 + i, N, residual_dtype)) for i, N in enumerate(widths)]
    x_ptr = gpu.to_device(x)
    width = np.dtype(cell[y_dtype]).itemsize
    outputs = [gpu.alloc(M * N * width + 64) for N in widths]
    try:
        results = []
        for how in (forced, "11,4", "4,1"):
            print(f"blocks of pairs K={K} M={M} y={y_dtype} residual={residual_dtype} shift={shift} forced={how}", flush=True)
            force("q4_gemm", how)
            force("trace", "1")
            capfd.readouterr()
            targets = [(w, y + shift * width, r) for w, y, r in zip(weights, outputs, residuals)]
            gpu.q4_sequence(engine.make_calls([(targets, x_ptr, engine.F32, M, getattr(engine, y_dtype),
                                                getattr(engine, residual_dtype or "F32"))]))
            gpu.sync()
            printed = capfd.readouterr().err
            if how == forced:
                assert f"{rows // 8} fragments of pairs x {16 * tiles} columns" in printed
                assert f"{blocks * K // 128} steps each" in printed
            results.append([gpu.download(y + shift * width, (M, N), cell[y_dtype]) for y, N in zip(outputs, widths)])
        for here, same, other in zip(*results):
            assert np.array_equal(here.view(np.uint16), same.view(np.uint16)) and np.any(here != 0)
            if y_dtype == "BF16":
                here, other = ((v.astype(np.uint32) << 16).view(np.float32) for v in (here, other))
            here, other = here.astype(np.float64), other.astype(np.float64)
            # K products of one row, of values and of remainders, summed in another order; two roundings to 11 or 8 bits
            rounding = {"F32": 0.0, "F16": 2.0 ** -11, "BF16": 2.0 ** -8}[y_dtype]
            assert np.max(np.abs(here - other)) <= 2 * (K * 2.0 ** -24 + rounding) * np.max(np.abs(other))
    finally:
        for pointer in [x_ptr] + outputs + [r for r in residuals if r is not None]:
            gpu.free(pointer)
        for weight in weights:
            weight.destroy()


@pytest.mark.parametrize("forced", ["11,2", "12,1", "13,1", "13,2"])
@pytest.mark.parametrize("x_dtype,M", [("F32", 9), ("F32", 35), ("F32", 64), ("BF16", 17), ("BF16", 75)])
def test_rows_kernel_targets_and_converted_activations(engine, gpu, force, forced, x_dtype, M):
    """Three weights of unequal width as one launch, activations converted: each output equals the
    same weight's own call under the other GEMM kernels up to the order of the fp32 sums."""
    K, widths = 448, (272, 1002, 100)
    x32 = make_x(engine, 101, M, K)
    x = x32 if x_dtype == "F32" else bf16_bits(x32).reshape(M, K)
    kind, x_dtype = engine.META_BF16_PLANES, getattr(engine, x_dtype)
    weights = [gpu.q4_prepare(*engine.synth_q4_affine(102 + i, 0.02, N, K, kind), N, K, kind) for i, N in enumerate(widths)]
    biases = [gpu.to_device(engine.synth_normal_f32(110 + i, 1.0, N)) for i, N in enumerate(widths)]
    x_ptr = gpu.to_device(x)
    outputs = [gpu.alloc(M * N * 4) for N in widths]
    try:
        results = []
        targets = list(zip(weights, outputs, biases))
        for how, groups in ((forced, [targets]), ("4,1", [[t] for t in targets])):
            print(f"rows targets M={M} x={x_dtype} forced={how}", flush=True)
            force("q4_gemm", how)
            gpu.q4_sequence(engine.make_calls([(g, x_ptr, x_dtype, M, engine.F32, engine.F32, engine.RESIDUAL_IS_BIAS)
                                               for g in groups]))
            gpu.sync()
            results.append([gpu.download(p, (M, N), np.float32) for p, N in zip(outputs, widths)])
        for here, there in zip(*results):
            assert np.any(there != 0)
            # 448 products of one row summed in another order: 448 roundings of 2^-24 at most
            assert np.max(np.abs(here - there)) <= 448 * 2.0 ** -24 * np.max(np.abs(there))
    finally:
        for pointer in [x_ptr] + outputs + biases:
            gpu.free(pointer)
        for weight in weights:
            weight.destroy()


@pytest.mark.parametrize("forced", ["11,2", "12,2", "11,1"])
@pytest.mark.parametrize("x_dtype,M", [("F16", 20), ("F16", 67), ("F32", 40), ("BF16", 128)])
def test_rows_kernel_runs_that_cross_targets(engine, gpu, force, forced, x_dtype, M):
    """Runs of steps that begin in one weight and end in the next, in blocks that other workgroups
    share: five steps a block in runs of three over 10, 16 and 6 blocks of 64 columns ("11,2") and in
    runs of two over 5, 8 and 3 of 128 ("12,2"), so that 50, 130, 25 and 65 steps precede a weight.  One width is no
    multiple of 4, the last weight's last block has tiles beyond the matrix.  Under "11,1" every
    workgroup takes whole blocks and a weight's outputs do not depend on the others, bit for bit."""
    K, widths = 640, (640, 1002, 330)
    x32 = make_x(engine, 131, M, K)
    x = x32 if x_dtype == "F32" else x32.astype(np.float16) if x_dtype == "F16" else bf16_bits(x32).reshape(M, K)
    kind, x_dtype = engine.META_BF16_PLANES, getattr(engine, x_dtype)
    weights = [gpu.q4_prepare(*engine.synth_q4_affine(132 + i, 0.02, N, K, kind), N, K, kind) for i, N in enumerate(widths)]
    x_ptr = gpu.to_device(x)
    outputs = [gpu.alloc(M * N * 4) for N in widths]
    try:
        results = []
        targets = list(zip(weights, outputs))
        for how, groups in ((forced, [targets]), ("11,1" if forced == "11,1" else "4,1", [[t] for t in targets])):
            print(f"rows across targets M={M} x={x_dtype} forced={how}", flush=True)
            force("q4_gemm", how)
            gpu.q4_sequence(engine.make_calls([(g, x_ptr, x_dtype, M, engine.F32) for g in groups]))
            gpu.sync()
            results.append([gpu.download(p, (M, N), np.float32) for p, N in zip(outputs, widths)])
        for here, there in zip(*results):
            assert np.any(there != 0)
            if forced == "11,1":
                assert np.array_equal(here, there)
            # 640 products of one row summed in another order: 640 roundings of 2^-24 at most
            assert np.max(np.abs(here - there)) <= 640 * 2.0 ** -24 * np.max(np.abs(there))
    finally:
        for pointer in [x_ptr] + outputs:
            gpu.free(pointer)
        for weight in weights:
            weight.destroy()


@pytest.mark.parametrize("M", [20, 150])
def test_targets_that_depend_on_each_other(engine, gpu, M):
    """A call whose second target adds the first one's output runs its targets in order: the same bits as one call per weight."""
    K = N = 256
    kind = engine.META_BF16_PLANES
    weights = [gpu.q4_prepare(*engine.synth_q4_affine(120 + i, 0.02, N, K, kind), N, K, kind) for i in range(2)]
    x = make_x(engine, 122, M, K).astype(np.float16)
    x_ptr, first, second = gpu.to_device(x), gpu.alloc(M * N * 2), gpu.alloc(M * N * 2)
    try:
        results = []
        targets = [(weights[0], first, None), (weights[1], second, first)]
        for groups in ([targets], [[t] for t in targets]):
            print(f"gemm dependent targets M={M} calls={len(groups)}", flush=True)
            gpu.q4_sequence(engine.make_calls([(g, x_ptr, engine.F16, M, engine.F16, engine.F16) for g in groups]))
            gpu.sync()
            results.append([gpu.download(p, (M, N), np.uint16) for p in (first, second)])
        for together, alone in zip(*results):
            assert np.array_equal(together, alone) and np.any(alone != 0)
    finally:
        for pointer in (x_ptr, first, second):
            gpu.free(pointer)
        for weight in weights:
            weight.destroy()


@pytest.mark.parametrize("forced", ["0,1", "0,2", "1,2", "3,1", "3,2", "5,2"])
@pytest.mark.parametrize("x_dtype,y_dtype,N", [("F32", "F32", 1101), ("BF16", "F16", 1104)])
def test_converted_activations_in_every_shape(engine, oracle, gpu, force, forced, x_dtype, y_dtype, N):
    """The first GEMM kernel's form for converted activations, in the shapes the test above leaves
    out: its own epilogue and partial sums, a last block of rows partly filled."""
    force("q4_gemm", forced)
    run_case(engine, oracle, gpu, N, 256, 75, engine.META_BF16_PLANES, getattr(engine, x_dtype), getattr(engine, y_dtype))


@pytest.mark.parametrize("splits", [2, 3, 4, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("N,x_dtype,y_dtype", [(1104, "F16", "F16"), (1101, "F16", "F32"), (1104, "F32", "F32"), (1101, "BF16", "F16")])
def test_k_split_sums(engine, oracle, gpu, force, splits, N, x_dtype, y_dtype):
    """The kernel behind a K split: every number of splits it is compiled for and one that it counts
    itself, four columns a thread and one, with and without rows that were converted."""
    force("q4_gemm", f"4,{splits}")
    run_case(engine, oracle, gpu, N, 1152, 75, engine.META_BF16_PLANES, getattr(engine, x_dtype), getattr(engine, y_dtype),
             residual=splits % 2 == 0)


@pytest.mark.parametrize("splits", [2, 9])
def test_k_split_sums_of_many_rows(engine, oracle, gpu, force, splits):
    """More rows than a grid's second dimension holds (65535)."""
    force("q4_gemm", f"0,{splits}")
    run_case(engine, oracle, gpu, 20, 1152, 65600, engine.META_BF16_PLANES, engine.F16, engine.F32)


@pytest.mark.parametrize("forced", ["6,2", "7,3", "8,2"])
@pytest.mark.parametrize("N", [1101, 1102, 1104])
@pytest.mark.parametrize("x_dtype,M", [("F16", 150), ("F32", 75), ("BF16", 128)])
def test_pipelined_k_split_of_any_width(engine, oracle, gpu, force, forced, N, x_dtype, M):
    """The pipelined kernel's partial sums are rows of 16-byte pieces whatever the width: padded
    columns, a last block of columns and of rows that is partly filled."""
    force("q4_gemm", forced)
    run_case(engine, oracle, gpu, N, 1152, M, engine.META_BF16_PLANES, getattr(engine, x_dtype), engine.F32, residual=M == 75)


@pytest.mark.parametrize("forced", ["6,1", "7,1", "8,1"])
@pytest.mark.parametrize("N", [1100, 1102, 1104])
@pytest.mark.parametrize("y_dtype", ["F16", "F32", "BF16"])
@pytest.mark.parametrize("M", [128, 150])
def test_pipelined_outputs_of_any_width(engine, oracle, gpu, force, forced, N, y_dtype, M):
    """The pipelined kernel's outputs of fp16 activations without a residual: rows that start on 16
    bytes, on 8 and on neither, blocks of columns and of rows that are whole and partly filled."""
    force("q4_gemm", forced)
    kind, K = engine.META_BF16_PLANES, 256
    quants, meta_a, meta_b = engine.synth_q4_affine(141, 0.02, N, K, kind)
    x = make_x(engine, 142, M, K).astype(np.float16)
    product = oracle.q4_linear(quants, meta_a, meta_b, kind, N, K, x, oracle.X_F16, M, weight_rounding=oracle.W_ROUND_F16)
    weight = gpu.q4_prepare(quants, meta_a, meta_b, N, K, kind)
    try:
        print(f"gemm outputs N={N} M={M} y={y_dtype} forced={forced}", flush=True)
        y = gpu.q4_linear(weight, x, engine.F16, getattr(engine, y_dtype))
        y = (y.astype(np.uint32) << 16).view(np.float32) if y_dtype == "BF16" else y
        # a bf16 output is rounded by at most half a unit of its eight bits: 2^-8 of its value
        assert q4_relative_error(y, product) <= (2.0 ** -8 if y_dtype == "BF16" else 1e-3)
    finally:
        weight.destroy()


@pytest.mark.parametrize("N,K,M,kernel", [(17408, 5120, 32, "rows"),    # 22.5 us from HBM; the other kernel 25.3
                                          (17408, 5120, 80, "rows"), (5120, 17408, 32, "rows"),
                                          (5120, 17408, 96, "rows"),    # 33.4, 37.9
                                          (5120, 6144, 32, "rows"),
                                          (17408, 5120, 112, "gemm"),   # 41.0, the other kernel 36.8
                                          (13758, 5312, 84, "rows")])   # 25.6, 33.4
def test_kernel_of_one_large_weight(engine, gpu, force, capfd, N, K, M, kernel):
    """Which kernel takes a large weight alone, as the trace prints it: the ones that timing each
    with weights in HBM and in the Infinity Cache found faster."""
    kind = engine.META_BF16_PLANES
    weight = gpu.q4_prepare(*engine.synth_q4_affine(151, 0.02, N, K, kind), N, K, kind)
    try:
        force("trace", "1")
        y = gpu.q4_linear(weight, make_x(engine, 152, M, K).astype(np.float16), engine.F16, engine.F16)
        printed = capfd.readouterr().err
    finally:
        weight.destroy()
    assert np.any(y != 0) and ("mi355q: q4 %s M=%d" % (kernel, M)) in printed


@pytest.mark.parametrize("forced", [None, "0,1", "1,2", "2,1", "3,3", "4,2", "5,1", "6,1", "6,3", "7,2", "8,1"])
@pytest.mark.parametrize("x_dtype,y_dtype,M", [("F16", "F16", 130), ("F16", "F32", 257), ("BF16", "BF16", 300), ("F32", "F32", 81)])
def test_targets_in_one_launch(engine, gpu, force, forced, x_dtype, y_dtype, M):
    """Weights of one call in one launch of the GEMM kernels: each output has the bits of its weight's
    own call.  Numbers of blocks that are and are not multiples of eight, ragged last tiles, a width that
    is no multiple of 4, fewer blocks than XCDs, more weights than one with and without a K split."""
    K, widths = 3072, (1280, 1002, 64, 100)
    x32 = make_x(engine, 141, M, K)
    x = x32 if x_dtype == "F32" else x32.astype(np.float16) if x_dtype == "F16" else bf16_bits(x32).reshape(M, K)
    kind, x_dtype, y_dtype = engine.META_BF16_PLANES, getattr(engine, x_dtype), getattr(engine, y_dtype)
    cell = np.uint32 if y_dtype == engine.F32 else np.uint16
    weights = [gpu.q4_prepare(*engine.synth_q4_affine(142 + i, 0.02, N, K, kind), N, K, kind) for i, N in enumerate(widths)]
    biases = [gpu.to_device(engine.synth_normal_f32(150 + i, 1.0, N)) for i, N in enumerate(widths)]
    x_ptr = gpu.to_device(x)
    outputs = [gpu.alloc(M * N * np.dtype(cell).itemsize) for N in widths]
    if forced:
        force("q4_gemm", forced)
    try:
        results = []
        targets = list(zip(weights, outputs, biases))
        for groups in ([targets[::-1]], [targets[:2], targets[2:]], [[t] for t in targets]):
            print(f"gemm one launch M={M} x={x_dtype} forced={forced} calls={len(groups)}", flush=True)
            for pointer, N in zip(outputs, widths):
                gpu.upload(pointer, np.full((M, N), 0x7FFF, cell))
            gpu.q4_sequence(engine.make_calls([(g, x_ptr, x_dtype, M, y_dtype, engine.F32, engine.RESIDUAL_IS_BIAS)
                                               for g in groups]))
            gpu.sync()
            results.append([gpu.download(p, (M, N), cell) for p, N in zip(outputs, widths)])
        for one, two, alone in zip(*results):
            assert np.any(alone != 0) and not np.any(alone == 0x7FFF)
            assert np.array_equal(one, alone) and np.array_equal(two, alone)
    finally:
        for pointer in [x_ptr] + outputs + biases:
            gpu.free(pointer)
        for weight in weights:
            weight.destroy()


@pytest.mark.parametrize("x_dtype,y_dtype,M,K,widths,moved", [
    ("F16", "F16", 200, 3072, (17408, 64), True),           # no split beside three, first kernel -> pipelined
    ("F16", "F32", 512, 5120, (6144, 1024, 1024), True),    # two splits beside four
    ("BF16", "BF16", 300, 3072, (6144, 102), False),        # a width that is no multiple of 4
    ("F16", "F32", 300, 1088, (5120, 64), False),           # K an odd multiple of 64
    ("F32", "F32", 130, 2112, (5120, 64), False),           # the same, pairs of rows
    ("F32", "F16", 200, 1600, (5120, 100, 64), True)])      # three weights, 17 tiles alone
def test_targets_whose_plans_differ(engine, gpu, force, capfd, x_dtype, y_dtype, M, K, widths, moved):
    """Weights of one launch whose own plans have different K splits, and (moved) another shape or kernel than the
    launch they share: the bits of each weight's own call, in both orders, with full residual rows."""
    x32 = make_x(engine, 181, M, K)
    x = x32 if x_dtype == "F32" else x32.astype(np.float16) if x_dtype == "F16" else bf16_bits(x32).reshape(M, K)
    kind, x_dtype, y_dtype = engine.META_BF16_PLANES, getattr(engine, x_dtype), getattr(engine, y_dtype)
    cell = np.uint32 if y_dtype == engine.F32 else np.uint16
    weights = [gpu.q4_prepare(*engine.synth_q4_affine(182 + i, 0.02, N, K, kind), N, K, kind) for i, N in enumerate(widths)]
    residuals = [gpu.to_device(engine.synth_normal_f32(190 + i, 1.0, M * N)) for i, N in enumerate(widths)]
    x_ptr = gpu.to_device(x)
    outputs = [gpu.alloc(M * N * np.dtype(cell).itemsize) for N in widths]
    force("trace", "1")
    try:
        results, plans = [], []
        targets = list(zip(weights, outputs, residuals))
        for groups in ([targets], [targets[::-1]], [[t] for t in targets]):
            print(f"gemm differing plans M={M} K={K} widths={widths} calls={len(groups)}", flush=True)
            for pointer, N in zip(outputs, widths):
                gpu.upload(pointer, np.full((M, N), 0x7FFF, cell))
            capfd.readouterr()
            gpu.q4_sequence(engine.make_calls([(g, x_ptr, x_dtype, M, y_dtype, engine.F32) for g in groups]))
            gpu.sync()
            printed = capfd.readouterr().err
            plans.append([(int(v), int(s), same != "") for v, s, same in
                          re.findall(r"q4 gemm .* -> variant (\d+) .*, K split (\d+)(, same launch)?\n", printed)])
            results.append([gpu.download(p, (M, N), cell) for p, N in zip(outputs, widths)])
    finally:
        for pointer in [x_ptr] + outputs + residuals:
            gpu.free(pointer)
        for weight in weights:
            weight.destroy()
    together, reverse, alone = plans
    assert [p[2] for p in together] == [False] + [True] * (len(widths) - 1) and not any(p[2] for p in alone)
    assert [p[1] for p in together] == [p[1] for p in alone] == [p[1] for p in reverse[::-1]]
    assert len({p[1] for p in alone}) > 1 and any(p[0] != together[0][0] for p in alone) == moved
    for one, other, by_itself in zip(*results):
        assert np.any(by_itself != 0) and not np.any(by_itself == 0x7FFF)
        assert np.array_equal(one, by_itself) and np.array_equal(other, by_itself)


@pytest.mark.parametrize("K", [3072, 1280])
def test_targets_in_one_launch_replayed(engine, gpu, K):
    """Shared launches, their conversion and the sums behind their K splits from a recorded graph: every replay, with
    eager calls of other sizes and new inputs between them, has the bits of the eager calls.  At 1280 columns the fp32
    call goes out by two kernels on one conversion."""
    kind = engine.META_BF16_PLANES
    weights = [gpu.q4_prepare(*engine.synth_q4_affine(201 + i, 0.02, N, K, kind), N, K, kind) for i, N in enumerate((6144, 100, 1001))]
    shapes = [(300, engine.F16, np.float16), (150, engine.F32, np.float32)]
    x_ptrs = [gpu.alloc(M * K * 4) for M, _, _ in shapes]
    outputs = [[gpu.alloc(M * w.N * 4) for w in weights] for M, _, _ in shapes]
    calls = engine.make_calls([(list(zip(weights, ys)), x, dtype, M, engine.F32)
                               for (M, dtype, _), x, ys in zip(shapes, x_ptrs, outputs)])
    other = engine.make_calls([([(weights[1], outputs[0][1])], x_ptrs[0], engine.F16, 40, engine.F32)])

    def fill(seed):
        for (M, _, cell), pointer in zip(shapes, x_ptrs):
            gpu.upload(pointer, make_x(engine, seed, M, K).astype(cell))

    def downloaded():
        gpu.sync()
        return [gpu.download(y, (M, w.N), np.uint32) for (M, _, _), ys in zip(shapes, outputs) for w, y in zip(weights, ys)]

    fill(1)
    graph = gpu.q4_sequence_record(calls)
    try:
        for replay in range(4):
            print(f"replay {replay} of shared launches", flush=True)
            fill(10 + replay)
            gpu.q4_sequence(calls)
            eager = downloaded()
            gpu.q4_sequence(other)
            gpu.graph_launch(graph)
            for one, two in zip(eager, downloaded()):
                assert np.any(one != 0) and np.array_equal(one, two)
    finally:
        gpu.graph_destroy(graph)
        for pointer in x_ptrs + outputs[0] + outputs[1]:
            gpu.free(pointer)
        for weight in weights:
            weight.destroy()


@pytest.mark.parametrize("forced", ["7,1", "7,3"])
def test_load_forms_of_targets_in_one_launch(engine, gpu, force, forced):
    """The 17-tile shape for several weights, like the one for one weight, gives the same bits with hand-scheduled and
    with compiler-managed weight loads, and those of each weight alone."""
    K, M, widths, kind = 1152, 260, (560, 1104), engine.META_BF16_PLANES
    weights = [gpu.q4_prepare(*engine.synth_q4_affine(171 + i, 0.02, N, K, kind), N, K, kind) for i, N in enumerate(widths)]
    x = make_x(engine, 173, M, K).astype(np.float16)
    force("q4_gemm", forced)
    try:
        print(f"gemm load forms of two weights forced={forced}", flush=True)
        scheduled = gpu.q4_linear_multi(weights, x, engine.F16, engine.F32)
        force("gemm_loads", "plain")
        plain = gpu.q4_linear_multi(weights, x, engine.F16, engine.F32)
        alone = [gpu.q4_linear(w, x, engine.F16, engine.F32) for w in weights]
    finally:
        for weight in weights:
            weight.destroy()
    for one, other, by_itself in zip(scheduled, plain, alone):
        assert np.any(by_itself != 0)
        assert np.array_equal(one.view(np.uint32), by_itself.view(np.uint32))
        assert np.array_equal(other.view(np.uint32), by_itself.view(np.uint32))


@pytest.mark.parametrize("K", [64, 512, 576, 1024, 1088, 1536, 1600, 2048, 2112, 4096, 4160, 6144, 6208, 8192, 8256, 18432, 18496])
def test_row_lengths_of_converted_activations(engine, oracle, gpu, K):
    """The conversion's forms by row length (a wave or a workgroup a row, so many columns a thread, a row
    read twice): five rows, whose largest value is the first, the last, or stands in the last octet but one."""
    N, M, kind = 16, 5, engine.META_BF16_PLANES
    quants, meta_a, meta_b = engine.synth_q4_affine(161, 0.02, N, K, kind)
    x = make_x(engine, 162, M, K).copy()
    x[0, 0], x[1, K - 1], x[2, K - 9], x[4] = 1e5, -3e6, 2e5, 0.0
    weight = gpu.q4_prepare(quants, meta_a, meta_b, N, K, kind)
    try:
        print(f"converted rows K={K}", flush=True)
        y = gpu.q4_linear(weight, x, engine.F32, engine.F32)
        y_bf = gpu.q4_linear(weight, bf16_bits(x).reshape(M, K), engine.BF16, engine.F32)
        rows = gpu.q4_dequant_rows(weight, np.arange(N, dtype=np.uint32))
    finally:
        weight.destroy()
    exact_rows = oracle.q4_linear(quants, meta_a, meta_b, kind, N, K, bf16_bits(x).reshape(M, K), oracle.X_BF16, M)
    # five fp32 rows are ten rows of the streaming kernel, which keeps the weight exact
    exact = oracle.q4_linear(quants, meta_a, meta_b, kind, N, K, x, oracle.X_F32, M)
    assert q4_relative_error(y[:4], exact[:4]) <= 1e-3 and q4_relative_error(y_bf[:4], exact_rows[:4]) <= 1e-3
    # value and remainder keep a row's numbers to 2^-22 of its largest, whose errors add like noise: 8 of that scale
    # at most.  Without the remainders the oracle's row without outliers is 290 to 970 of it off
    scale = 2.0 ** -22 * np.abs(x).max(axis=1, keepdims=True) * np.sqrt(np.sum(rows.astype(np.float64) ** 2, axis=1))
    assert np.all(np.abs(y[:4] - exact[:4]) <= 8.0 * scale[:4])
    assert np.all(y[4] == 0.0) and np.all(y_bf[4] == 0.0)
