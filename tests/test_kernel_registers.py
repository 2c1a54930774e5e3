"""Registers that the built kernels spill, read from the metadata of the code objects in the library."""

import struct

import pytest

from blksprs_amd.csrc.build import LIB

msgpack = pytest.importorskip("msgpack")

EM_AMDGPU, SHT_NOTE, NT_AMDGPU_METADATA = 224, 7, 32


def _kernels(image: bytes):
    """Metadata of the kernels of every AMDGPU code object inside ``image``."""
    at = image.find(b"\x7fELF", 4)
    while at >= 0:
        if struct.unpack_from("<H", image, at + 18)[0] == EM_AMDGPU:
            sections, = struct.unpack_from("<Q", image, at + 40)
            size, count = struct.unpack_from("<HH", image, at + 58)
            for i in range(count):
                _, kind, _, _, offset, length = struct.unpack_from("<IIQQQQ", image, at + sections + i * size)
                while kind == SHT_NOTE and length > 0:
                    n_name, n_desc, note = struct.unpack_from("<III", image, at + offset)
                    name_end = offset + 12 + (n_name + 3) // 4 * 4
                    if note == NT_AMDGPU_METADATA:
                        yield from msgpack.unpackb(image[at + name_end:at + name_end + n_desc])["amdhsa.kernels"]
                    step = name_end + (n_desc + 3) // 4 * 4 - offset
                    offset, length = offset + step, length - step
        at = image.find(b"\x7fELF", at + 4)


@pytest.fixture(scope="module")
def kernels():
    if not LIB.exists():
        pytest.skip("library not built")
    return {k[".name"]: k for k in _kernels(LIB.read_bytes())}


@pytest.mark.parametrize("kernel", ["fwd", "dq", "dkv"])
@pytest.mark.parametrize("slices,halves", [(1, 1), (2, 1), (3, 1), (4, 1), (2, 2), (4, 2)])
def test_fp32_attention_keeps_its_registers(kernels, kernel, slices, halves):
    """Blocks of 32 (halves 1) and of 64 (2).  dK / dV: up to two at head dimension 64 in halves, stored once in front of the walk; at 128
    operands in parts and sums take 320 of 512 registers and up to 28 of the rest are stored and loaded in a step of 3100
    instructions."""
    found = [k for name, k in kernels.items()
             if f"attn_small_{kernel}_kernelI" in name and f"SF32ELi32ELi{slices}ELb0ELi{halves}EE" in name]
    assert len(found) == 1
    spilled = found[0][".vgpr_spill_count"]
    assert spilled <= ({(2, 2): 2, (4, 1): 28, (4, 2): 28}.get((slices, halves), 0) if kernel == "dkv" else 0)


@pytest.mark.parametrize("kernel", ["fwd", "dq", "dkv"])
@pytest.mark.parametrize("sbs,most", [(16, 8), (32, 4)])
def test_16_bit_attention_of_small_blocks_keeps_its_registers(kernels, kernel, sbs, most):
    """Every head dimension, with and without slices that may be missing."""
    found = [k for name, k in kernels.items() if f"attn_small_{kernel}_kernelI" in name and f"ELi{sbs}ELi" in name and "SF32" not in name]
    assert len(found) == 2 * 2 * most
    assert all(k[".vgpr_spill_count"] == 0 for k in found)
