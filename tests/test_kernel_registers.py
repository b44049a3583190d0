"""Registers that spill to memory, as the compiler notes them beside the kernels of a built library: the loops of these kernels are
written for what a wave's registers hold, and a change far from a loop (a sum behind it) can push it out of them."""
import struct

import msgpack
import pytest

from arle_amd.kernels import build

_NOTE, _AMDGPU_METADATA = 7, 32      # section type of notes; type of the note that lists the kernels


def _code_objects(data: bytes):
    """The GPU's ELF files inside a library: every entry for the GPU of every bundle."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    start = data.find(magic)
    while start >= 0:
        (count,), at = struct.unpack_from("<Q", data, start + len(magic)), start + len(magic) + 8
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", data, at)
            triple = data[at + 24:at + 24 + name]
            at += 24 + name
            if b"amdgcn" in triple and size:
                yield data[start + offset:start + offset + size]
        start = data.find(magic, start + len(magic))


def _kernels(elf: bytes) -> dict:
    """Mangled name -> the compiler's note of a kernel."""
    found = {}
    sections, = struct.unpack_from("<Q", elf, 0x28)
    entry, count = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        _, kind, _, _, at, size = struct.unpack_from("<IIQQQQ", elf, sections + i * entry)
        end = at + size
        while kind == _NOTE and at < end:
            name, length, note = struct.unpack_from("<III", elf, at)
            at += 12 + -(-name // 4) * 4
            if note == _AMDGPU_METADATA:
                found.update((k[".name"], k) for k in msgpack.unpackb(elf[at:at + length], strict_map_key=False)["amdhsa.kernels"])
            at += -(-length // 4) * 4
    return found


@pytest.fixture(scope="module")
def softcap() -> dict:
    with open(build.ensure("attention_softcap"), "rb") as fh:
        data = fh.read()
    found = {}
    for elf in _code_objects(data):
        found.update(_kernels(elf))
    assert found
    return found


# (chunks of the key size, of the value size, a decoded row's heads, waves, blocks of rows): the most registers that may spill
@pytest.mark.parametrize("form,most", [
    *(((4, 8, 0, waves, 2), 0) for waves in (1, 2, 4)),       # portions of heads up to 128, 32 rows a wave
    *(((4, 8, 0, waves, 1), 0) for waves in (1, 2, 4)),
    ((4, 8, 1, 8, 1), 1),                                     # decoded rows
    ((8, 12, 1, 8, 1), 25), ((8, 16, 1, 8, 1), 69),           # ... of more columns than two waves a SIMD have registers for
])
def test_the_soft_capped_kernels_stay_in_their_registers(softcap, form, most):
    kc, vc, heads, waves, blocks = form
    name = f"attn_softcap_mfma_kernelILi{kc}ELi{vc}ELb{heads}ELi{waves}ELi{blocks}E"
    notes = [k for n, k in softcap.items() if name in n]
    assert len(notes) == 1
    assert notes[0][".vgpr_spill_count"] <= most


def test_the_shared_tiles_of_soft_capped_portions_stay_in_their_registers(softcap):
    notes = [k for n, k in softcap.items() if "cap_portions_kernel" in n]
    assert len(notes) == 3 and all(k[".vgpr_spill_count"] == 0 and k[".vgpr_count"] <= 256 for k in notes)
