"""What the compiler gave the kernels, read from the built library: the hot kernels keep nothing of a lane in memory."""

import re
import struct
import subprocess
from pathlib import Path

import msgpack
import pytest


def _images(data):
    """Where the code objects embedded in the host library begin and end, their section headers and how many these are."""
    for image in re.finditer(b"\x7fELF\x02\x01\x01\x40", data):      # ELF64 of the AMDGPU HSA ABI
        at = image.start()
        sections, (size, count) = at + struct.unpack_from("<Q", data, at + 40)[0], struct.unpack_from("<HH", data, at + 58)
        yield at, sections + size * count, sections, size, count


def _kernels(path):
    """The kernels' entries of the code objects' metadata notes (msgpack), by mangled name."""
    data = path.read_bytes()
    found = {}
    for at, _, sections, size, count in _images(data):
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
def library():
    from llmx_amd.csrc import build
    return build.load_path()


@pytest.fixture(scope="module")
def kernels(library):
    return _kernels(library)


# decode attention, every head size, contexts walked (0) and shared out (1): heads of 224 to 256 once kept up to 349 registers a lane in memory
def test_decode_attention_keeps_its_registers(kernels):
    names = [f"paged_attention_mfma_kernelILi{dt}ELb{partial}E" for dt in range(1, 17) for partial in (0, 1)]
    for name in names:
        kernel = [k for n, k in kernels.items() if name in n]
        assert len(kernel) == 1, name
        assert kernel[0][".private_segment_fixed_size"] == 0, (name, kernel[0][".vgpr_spill_count"])


# the streaming products: those that add or have a bias a feature kept up to 20 registers a lane in memory
@pytest.mark.parametrize("kernel", ["gemm_skinny_kernel", "gemm_f32_stream_kernel"])
def test_streaming_products_keep_their_registers(kernel, kernels):
    found = {n: k for n, k in kernels.items() if kernel in n}
    assert len(found) > 20
    assert {n: k[".vgpr_spill_count"] for n, k in found.items() if k[".private_segment_fixed_size"]} == {}


# weights are asked for from a place the wave shares; where the compiler does not know it for one, each load becomes a loop over the lanes' places
@pytest.mark.parametrize("kernel", ["gemm_f32_stream_kernel", "gemm_skinny_kernel"])
def test_streamed_weights_are_asked_for_once(kernel, library, tmp_path):
    objdump = Path("/opt/rocm/llvm/bin/llvm-objdump")
    if not objdump.exists():
        pytest.skip("no disassembler")
    data, seen = library.read_bytes(), 0
    for i, (at, end, *_) in enumerate(_images(data)):
        if kernel.encode() not in data[at:end]:
            continue
        image = tmp_path / f"{i}.o"
        image.write_bytes(data[at:end])
        text = subprocess.run([str(objdump), "-d", str(image)], capture_output=True, text=True, check=True).stdout
        for name, body in re.findall(r"^[0-9a-f]+ <(\S+)>:\n(.*?)(?=^[0-9a-f]+ <|\Z)", text, re.M | re.S):
            if kernel in name and "buffer_load_dwordx4" in body:
                seen += 1
                assert body.count("v_readfirstlane") <= 4, name
    assert seen > 20
