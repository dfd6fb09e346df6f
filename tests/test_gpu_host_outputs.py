"""Outputs that leave for the caller's memory in chunks (512 KiB and more) are the bytes that the same call
leaves in device memory: at the smallest such output and one below it, at whole halves of the pinned memory
they pass through and one output beyond, at ends that are no multiple of 16 bytes, through each half more
than once, and for two calls one after the other; and so with every entry point that has them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HALF = 2 << 20


@pytest.mark.parametrize("N,M,y_dtype", [
    (4096, 32, "F32"),        # 512 KiB
    (4095, 32, "F32"),        # below: the runtime's own copy
    (1023, 513, "F16"),       # odd fp16 columns: the last chunk ends at 14 bytes of 16
    (4096, 128, "F32"),       # one half
    (HALF // 4 + 1, 1, "F32"),  # one half and 4 bytes
    (HALF // 2 - 3, 1, "F16"),  # one half less 6 bytes, one row
    (4097, 256, "F32"),       # two halves and 1 KiB
    (3001, 700, "BF16"),
    (2049, 1100, "F32"),      # five parts
])
def test_host_outputs_are_the_device_outputs(engine, gpu, N, M, y_dtype):
    K = 128
    kind = getattr(engine, y_dtype)
    cell = 4 if y_dtype == "F32" else 2
    quants, a, b = engine.synth_q4_affine(N + M, 0.02, N, K, engine.META_F16_INTERLEAVED)
    weight = gpu.q4_prepare(quants, a, b, N, K, engine.META_F16_INTERLEAVED)
    print(f"host outputs {M} x {N} {y_dtype}: {M * N * cell} bytes", flush=True)
    y_device = gpu.alloc(M * N * cell)
    x_device = gpu.alloc(M * K * 2)
    try:
        for seed in (1, 2):
            x = engine.synth_normal_f16(seed, 1.0, M * K).reshape(M, K)
            gpu.upload(x_device, x)
            gpu.q4_linear_device(weight, x_device, engine.F16, M, y_device, kind, asynchronous=False)
            expected = gpu.download(y_device, (M, N), np.uint32 if cell == 4 else np.uint16)
            got = gpu.q4_linear(weight, x, engine.F16, kind)
            assert np.array_equal(got.view(expected.dtype).reshape(M, N), expected)
    finally:
        gpu.free(y_device)
        gpu.free(x_device)
        weight.destroy()


def test_w8a8_outputs_leave_in_chunks(engine, gpu, force, capfd):
    """Every large output of a W8A8 call goes through the pinned chunks, whatever the sizes of those staged before
    it (odd widths and an odd number of rows: multiples of 4 bytes), accumulators too."""
    K, M, widths = 32, 331, (1001, 1003, 998)
    rows = [engine.synth_w8_rows(5 + i, 0.02, N, K) for i, N in enumerate(widths)]
    weights = [gpu.w8a8_prepare(r, N, K) for r, N in zip(rows, widths)]
    q, scales = gpu.quantize_i8(engine.synth_normal_f32(9, 1.0, M * K).reshape(M, K))
    biases = [engine.synth_normal_f32(20 + i, 1.0, N) for i, N in enumerate(widths)]
    pointers = [[gpu.alloc(M * N * 4) for N in widths] for _ in range(2)]
    on_device = [gpu.to_device(q), gpu.to_device(scales)] + [gpu.to_device(b) for b in biases]
    force("trace", "1")
    try:
        print(f"w8a8 host outputs {M} x {widths}", flush=True)
        capfd.readouterr()
        got = gpu.w8a8_linear_multi(weights, widths, q, scales, biases)
        printed = capfd.readouterr().err
        gpu.w8a8_linear_multi_device(weights, on_device[0], on_device[1], M, on_device[2:], *pointers)
        gpu.sync()
        expected = [[gpu.download(p, (M, N), np.uint32) for p, N in zip(kind, widths)] for kind in pointers]
    finally:
        for pointer in pointers[0] + pointers[1] + on_device:
            gpu.free(pointer)
        for weight in weights:
            gpu.w8a8_destroy(weight)
    for (out, acc), out_ref, acc_ref, N in zip(got, *expected, widths):
        assert np.any(acc_ref != 0)
        assert np.array_equal(out.view(np.uint32), out_ref) and np.array_equal(acc.view(np.uint32), acc_ref)
        assert printed.count(f"host outputs, {M * N * 4} bytes in chunks") == 2


def test_several_q4_outputs_leave_in_chunks(engine, gpu, force, capfd):
    """Outputs of one call one after the other through the same pinned halves: the first of more than one half, the
    second of two and more."""
    K, M, widths, kind = 128, 521, (1003, 2049), engine.META_F16_INTERLEAVED
    weights = [gpu.q4_prepare(*engine.synth_q4_affine(31 + i, 0.02, N, K, kind), N, K, kind) for i, N in enumerate(widths)]
    x = engine.synth_normal_f16(33, 1.0, M * K).reshape(M, K)
    x_ptr, pointers = gpu.to_device(x), [gpu.alloc(M * N * 4) for N in widths]
    force("trace", "1")
    try:
        for _ in range(2):
            print(f"q4 host outputs {M} x {widths}", flush=True)
            capfd.readouterr()
            got = gpu.q4_linear_multi(weights, x, engine.F16, engine.F32)
            printed = capfd.readouterr().err
            gpu.q4_sequence(engine.make_calls([(list(zip(weights, pointers)), x_ptr, engine.F16, M, engine.F32)]))
            gpu.sync()
            for y, pointer, N in zip(got, pointers, widths):
                assert np.array_equal(y.view(np.uint32), gpu.download(pointer, (M, N), np.uint32))
                assert printed.count(f"host outputs, {M * N * 4} bytes in chunks") == 1
    finally:
        for pointer in pointers + [x_ptr]:
            gpu.free(pointer)
        for weight in weights:
            weight.destroy()


@pytest.mark.parametrize("M", [12, 150])  # the streaming kernel's rows, the GEMM's
def test_q8_outputs_leave_in_chunks(engine, gpu, force, capfd, M):
    N, K = 16411, 128
    records = engine.synth_w8_rows(41, 0.02, N, K)
    weight = gpu.q8rows_prepare(records, N, K)
    x = engine.synth_normal_f16(42, 1.0, M * K).reshape(M, K)
    x_ptr, pointer = gpu.to_device(x), gpu.alloc(M * N * 4)
    force("trace", "1")
    try:
        print(f"q8 host outputs {M} x {N}", flush=True)
        capfd.readouterr()
        got = gpu.q8_linear(weight, N, x, engine.F16, engine.F32)
        printed = capfd.readouterr().err
        gpu.q8_linear_device(weight, x_ptr, engine.F16, M, pointer, engine.F32, asynchronous=False)
        assert np.array_equal(got.view(np.uint32), gpu.download(pointer, (M, N), np.uint32)) and np.any(got != 0)
        assert printed.count(f"host outputs, {M * N * 4} bytes in chunks") == 1
    finally:
        gpu.free(pointer)
        gpu.free(x_ptr)
        gpu.q8_destroy(weight)
