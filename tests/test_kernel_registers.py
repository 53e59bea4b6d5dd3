"""The registers of compiled kernels, as the built library's own metadata gives them: two waves share a SIMD's 512 only if
neither takes more than 256, and what a kernel loses with the second wave no comparison of results shows."""

import struct

import pytest

from bitwise_amd.csrc import build

msgpack = pytest.importorskip("msgpack")
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def kernels():
    """name -> metadata of every gfx950 kernel of the built library."""
    lib = build._find_current()
    if lib is None:
        pytest.skip("the kernel library is not built")
    data, out, at = lib.read_bytes(), {}, -1
    while (at := data.find(BUNDLE, at + 1)) >= 0:
        entry = at + len(BUNDLE) + 8
        for _ in range(struct.unpack_from("<Q", data, at + len(BUNDLE))[0]):
            offset, size, n = struct.unpack_from("<QQQ", data, entry)
            if data[entry + 24:entry + 24 + n].endswith(b"gfx950"):
                out.update(code_object_kernels(data[at + offset:at + offset + size]))
            entry += 24 + n
    return out


def code_object_kernels(elf):
    headers, (size, count) = struct.unpack_from("<Q", elf, 0x28)[0], struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        kind, _, _, offset, length = struct.unpack_from("<IQQQQ", elf, headers + i * size + 4)
        if kind == 7:                                        # a note section: name size, value size, type, name, value
            name, value = struct.unpack_from("<II", elf, offset)
            start = offset + 12 + (name + 3) // 4 * 4
            return {k[".name"]: k for k in msgpack.unpackb(elf[start:start + value])["amdhsa.kernels"]}
    return {}


@pytest.mark.parametrize("mode", [1, 3, 4, 5])
@pytest.mark.parametrize("dim", [16, 32, 64, 128, 256])
def test_memory_walk_leaves_room_for_a_second_wave(mode, dim):
    """The walk of a portion (memories with scalar gates, a constant decay, a step size, the delta rule)."""
    found = [k for name, k in kernels().items() if f"linear_recurrence_kernelILi{mode}ELi{dim}ELi0E" in name]
    assert len(found) == 1
    assert found[0][".vgpr_count"] <= 256          # (accumulation registers included)


def test_norm_with_shift_leaves_room_for_four_waves():
    """Four waves of up to 128 registers share a SIMD; with both rows kept in registers the kernel took 142, three waves."""
    found = [k for name, k in kernels().items() if "norm_shift_kernelI" in name]
    assert len(found) == 2
    assert all(k[".vgpr_count"] <= 128 for k in found)
