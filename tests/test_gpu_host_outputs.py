"""Outputs that leave for the caller's memory in chunks (512 KiB and more) are the bytes that the same call
leaves in device memory: at the smallest such output and one below it, at whole halves of the pinned memory
they pass through and one output beyond, at ends that are no multiple of 16 bytes, through each half more
than once, and for two calls one after the other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HALF = 2 << 20


@pytest.mark.parametrize("N,M,y_dtype", [
    (4096, 32, "F32"),        # 512 KiB
    (4095, 32, "F32"),        # below: the runtime's own copy
    (1023, 513, "F16"),       # odd fp16 columns: the last chunk ends at 2 bytes of 16
    (4096, 128, "F32"),       # one half
    (HALF // 4 + 1, 1, "F32"),  # one half and 4 bytes
    (HALF // 2 - 3, 1, "F16"),  # half a half less 6 bytes, one row
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
