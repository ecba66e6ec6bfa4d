"""What the built kernels take of a compute unit's registers, read from the notes of the built library's code objects (no
GPU): products whose times rest on two blocks a unit, or on nothing kept in memory, keep to it."""
import re
import struct

import pytest


def kernels(name):
    """[(kernel's name, its metadata)] of a kernel library built from this tree's sources."""
    import msgpack
    from allpaca_amd.kernels import build
    with open(build.build(name, verbose=False), "rb") as f:
        data = f.read()
    found = []
    for at in [m.start() for m in re.finditer(rb"__CLANG_OFFLOAD_BUNDLE__", data)]:
        count, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(count):
            offset, size, n = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + n].decode()
            p += 24 + n
            if "gfx950" in target and size:
                found += notes(data[at + offset:at + offset + size], msgpack)
    assert found
    return found


def notes(elf, msgpack):
    assert elf[:5] == b"\x7fELF\x02"
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    entry, count = struct.unpack_from("<HH", elf, 0x3A)
    out = []
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, shoff + i * entry + 4)
        offset, size = struct.unpack_from("<QQ", elf, shoff + i * entry + 24)
        if kind != 7:                                        # SHT_NOTE
            continue
        p = offset
        while p < offset + size:
            n, d, what = struct.unpack_from("<III", elf, p)
            body = p + 12 + -(-n // 4) * 4
            if what == 32:                                   # NT_AMDGPU_METADATA
                meta = msgpack.unpackb(elf[body:body + d], raw=False, strict_map_key=False)
                out += [(k[".name"], k) for k in meta["amdhsa.kernels"]]
            p = body + -(-d // 4) * 4
    return out


def arguments(name, kernel):
    """The template arguments of a kernel's mangled name, or None."""
    m = re.search(kernel + r"I((?:L[ib]\d+E)+)", name)
    return tuple(int(v) for v in re.findall(r"L[ib](\d+)E", m.group(1))) if m else None


def test_products_of_few_rows_keep_their_registers():
    pytest.importorskip("msgpack")
    seen = 0
    for name, k in kernels("tuned"):
        args = arguments(name, "skinny_gemm_kernel")
        if args is None:
            continue
        groups, mode, bands, waves, pre, emit = args
        seen += 1
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, args
        if waves == 8 and (mode == 3 or (bands == 1 and pre)):   # 3: SwiGLU.  Two blocks of 8 waves a unit
            assert k[".vgpr_count"] <= 128, args
    assert seen >= 80


def test_products_of_17_to_64_rows_keep_nothing_in_memory():
    pytest.importorskip("msgpack")
    found = [(arguments(name, "rows_gemm_kernel"), k) for name, k in kernels("tuned")]
    found = [(args, k) for args, k in found if args]
    assert len(found) >= 80
    for args, k in found:
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, args


def test_adding_kernels_leave_room_for_eight_waves_a_simd():
    """They are bound by loads in flight, of which a lane that takes its columns one by one has few."""
    pytest.importorskip("msgpack")
    found = [(arguments(name, kernel), k) for name, k in kernels("tuned")
             for kernel in ("gemm_finish_kernel", "gemm_finish_qkv_rope_kernel") if arguments(name, kernel)]
    assert len(found) >= 4
    for args, k in found:
        assert k[".vgpr_count"] <= 64 and k[".private_segment_fixed_size"] == 0, args
