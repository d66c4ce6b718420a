"""What the compiled kernels need, from the metadata of the code objects in the
built library: the sweeps and factorisations keep everything in registers (no
scratch memory per lane), and the small sweeps leave room for three waves per
SIMD (168 of its 512 registers each, in steps of eight)."""

import os
import struct

import msgpack
import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fd_adi_amd",
                   "libfdadi.so")


def _notes(elf):
    """(type, payload) of every note of a 64-bit little-endian ELF image."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    size, num = struct.unpack_from("<HH", elf, 0x3A)
    for k in range(num):
        kind, = struct.unpack_from("<I", elf, shoff + k * size + 4)
        off, length = struct.unpack_from("<QQ", elf, shoff + k * size + 0x18)
        at = off
        while kind == 7 and at < off + length:
            nlen, dlen, typ = struct.unpack_from("<III", elf, at)
            data = at + 12 + (nlen + 3) // 4 * 4
            yield typ, elf[data:data + dlen]
            at = data + (dlen + 3) // 4 * 4


def kernels():
    """Metadata of every kernel of the library, by its (mangled) name."""
    blob = open(LIB, "rb").read()
    out, magic, bundle = {}, b"\x7fELF\x02\x01\x01\x40", b"__CLANG_OFFLOAD_BUNDLE__"
    at = blob.find(bundle)
    while at >= 0:
        n, = struct.unpack_from("<Q", blob, at + 24)
        pos = at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, pos)
            pos += 24 + idlen
            elf = blob[at + off:at + off + size]
            if elf.startswith(magic):
                for typ, data in _notes(elf):
                    if typ == 32:  # AMDGPU metadata
                        for k in msgpack.unpackb(data)["amdhsa.kernels"]:
                            out[k[".name"]] = k
        at = blob.find(bundle, at + 1)
    return out


@pytest.mark.parametrize("name, least", [("spot_sweep_kernel", 80), ("var_sweep_kernel", 14),
                                         ("factor_kernel", 1), ("tri_solve_kernel", 2)])
def test_no_scratch(name, least):
    ks = {n: k for n, k in kernels().items() if name in n}
    assert len(ks) >= least
    bad = {n: (k[".private_segment_fixed_size"], k[".vgpr_spill_count"]) for n, k in ks.items()
           if k[".private_segment_fixed_size"] or k[".vgpr_spill_count"]}
    assert not bad


@pytest.mark.parametrize("mode", [0, 2])  # SM_FIRST and SM_CS, four columns, 8 rows
def test_three_waves(mode):
    ks = {n: k[".vgpr_count"] for n, k in kernels().items()
          if "spot_sweep_kernelILi%dE" % mode in n and "ELi4ELi8EEE" in n}
    assert len(ks) == 4 and max(ks.values()) <= 168, ks
