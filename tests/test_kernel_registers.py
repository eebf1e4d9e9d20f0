"""What the compiler gave the kernels, read from the built library: the hot kernels keep nothing of a lane in memory."""

import re
import struct

import msgpack
import pytest


def _kernels(path):
    """The kernels' entries of the code objects' metadata notes (msgpack), by mangled name."""
    data = path.read_bytes()
    found = {}
    for image in re.finditer(b"\x7fELF\x02\x01\x01\x40", data):      # ELF64 of the AMDGPU HSA ABI, embedded in the host library
        at = image.start()
        sections, (size, count) = at + struct.unpack_from("<Q", data, at + 40)[0], struct.unpack_from("<HH", data, at + 58)
        for s in range(count):
            kind, _, _, offset, length = struct.unpack_from("<IQQQQ", data, sections + s * size + 4)
            if kind != 7:       # SHT_NOTE
                continue
            name_size, note_size, note_kind = struct.unpack_from("<III", data, at + offset)
            if note_kind == 32:     # NT_AMDGPU_METADATA
                begin = at + offset + 12 + (name_size + 3) // 4 * 4
                found.update((k[".name"], k) for k in msgpack.unpackb(data[begin:begin + note_size])["amdhsa.kernels"])
    return found


@pytest.fixture(scope="module")
def kernels():
    from llmx_amd.csrc import build
    return _kernels(build.load_path())


# decode attention, every head size, contexts walked (0) and shared out (1): heads of 224 to 256 once kept up to 349 registers a lane in memory
def test_decode_attention_keeps_its_registers(kernels):
    names = [f"paged_attention_mfma_kernelILi{dt}ELb{partial}E" for dt in range(1, 17) for partial in (0, 1)]
    for name in names:
        kernel = [k for n, k in kernels.items() if name in n]
        assert len(kernel) == 1, name
        assert kernel[0][".private_segment_fixed_size"] == 0, (name, kernel[0][".vgpr_spill_count"])
