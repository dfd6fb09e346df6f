"""q4_rows_kernel (csrc/q4_rows_device.h) orders its waves' accesses to LDS by counted waits and barriers: in the built code they
are LDS accesses, not flat ones, which are counted with those to memory, too."""
import struct
import subprocess
from pathlib import Path

LIBRARY = Path(__file__).resolve().parent.parent / "cpu-llms-in-c_amd" / "lib" / "libmi355q.so"
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def device_images(data):
    """The device ELF images of the library, one for each source file."""
    at = data.find(MAGIC)
    while at >= 0:
        entries, = struct.unpack_from("<Q", data, at + len(MAGIC))
        here = at + len(MAGIC) + 8
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, here)
            name = data[here + 24:here + 24 + length]
            here += 24 + length
            if b"gfx950" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + 1)


def test_no_flat_accesses(tmp_path):
    images = [image for image in device_images(LIBRARY.read_bytes()) if b"q4_rows_kernel" in image]
    assert len(images) == 3  # blocks of 4, 8 and 16 tiles
    for number, image in enumerate(images):
        path = tmp_path / f"rows_{number}.co"
        path.write_bytes(image)
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], capture_output=True, text=True, check=True).stdout
        assert "v_mfma_f32_16x16x32_f16" in listing and "ds_read" in listing
        flat = [line.strip() for line in listing.splitlines() if "flat_load" in line or "flat_store" in line]
        assert not flat, flat[:5]
