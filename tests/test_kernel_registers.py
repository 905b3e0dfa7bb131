"""What the compiler reports of the built kernels (the metadata that it leaves in the library for the loader)."""
import struct

import msgpack
import pytest

from gpullama3_java_amd.csrc import build

AMDGPU, NOTE, METADATA = 224, 7, 32


def kernels():
    with open(build.library_path() or build.build(), "rb") as f:
        data = f.read()
    at = data.find(b"\x7fELF", 1)
    while at >= 0:
        machine, = struct.unpack_from("<H", data, at + 18)
        if machine == AMDGPU:
            sections, = struct.unpack_from("<Q", data, at + 40)
            size, count = struct.unpack_from("<HH", data, at + 58)
            for i in range(count):
                _, kind, _, _, offset = struct.unpack_from("<IIQQQ", data, at + sections + i * size)
                if kind == NOTE:
                    name, length, note = struct.unpack_from("<III", data, at + offset)
                    if note == METADATA:
                        first = at + offset + 12 + (name + 3) // 4 * 4
                        yield from msgpack.unpackb(data[first:first + length])["amdhsa.kernels"]
        at = data.find(b"\x7fELF", at + 1)


@pytest.mark.parametrize("name", ["attention_f32_kernel", "attention_prefill", "gemm_f32_", "gemm_mfma_"])
def test_kernels_whose_loads_wait_in_registers_have_the_registers(name):
    """Loads that are asked for ahead and do not fit go through scratch memory, which is slower than not asking ahead."""
    found = [k for k in kernels() if name in k[".name"]]
    assert found
    assert [k[".name"] for k in found if k[".private_segment_fixed_size"]] == []
