"""Resources of the built kernels, from the code object metadata of the library: the
batched kernels keep nothing in scratch memory (arrays that the compiler leaves
there also cost a wave per SIMD and are written once per item and lane)."""
import struct

import pytest

msgpack = pytest.importorskip("msgpack")


def _kernels():
    """Metadata of every gfx950 kernel of the library, by mangled name."""
    from mentpy_amd import _native as nat
    data = nat.LIB_PATH.read_bytes()
    found, at = {}, data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + n]
            p += 24 + n
            if b"gfx950" in name and size:
                found.update(_notes(data[at + off:at + off + size]))
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)
    return found


def _notes(elf):
    """amdhsa.kernels of a 64-bit little-endian code object."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    entry, count = struct.unpack_from("<HH", elf, 58)
    out = {}
    for i in range(count):
        _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + i * entry)
        if kind != 7:                       # SHT_NOTE
            continue
        p = off
        while p < off + size:
            nlen, dlen, _ = struct.unpack_from("<III", elf, p)
            d = p + 12 + (nlen + 3) // 4 * 4
            if elf[p + 12:p + 12 + nlen].rstrip(b"\0") == b"AMDGPU":
                for k in msgpack.unpackb(elf[d:d + dlen])["amdhsa.kernels"]:
                    out[k[".name"]] = k
            p = d + (dlen + 3) // 4 * 4
    return out


def test_batched_kernels_use_no_scratch():
    kernels = _kernels()
    if not kernels:
        pytest.skip("the library's code objects are not readable (compressed)")
    batched = {n: k for n, k in kernels.items() if "k_batch_mixed" in n or "7k_batchI" in n}
    assert sum("k_batch_mixed" in n for n in batched) == 8
    bad = {n: k[".private_segment_fixed_size"] for n, k in batched.items()
           if k[".private_segment_fixed_size"]}
    assert not bad
