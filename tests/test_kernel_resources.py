"""Registers of the built library's kernels, from the metadata of its code objects."""
import struct

import pytest


def _kernels(path):
    """name -> metadata of every kernel in the library's embedded gfx950 code objects (ELF files with
    a msgpack note of owner AMDGPU)."""
    msgpack = pytest.importorskip("msgpack")
    data, out, at = path.read_bytes(), {}, 0
    while True:
        at = data.find(b"\x7fELF\x02\x01", at + 1)  # from 1: the library itself is one too
        if at < 0:
            return out
        if struct.unpack_from("<H", data, at + 18)[0] != 224:  # EM_AMDGPU
            continue
        phoff, phnum = struct.unpack_from("<Q", data, at + 32)[0], struct.unpack_from("<H", data, at + 56)[0]
        for i in range(phnum):
            kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", data, at + phoff + 56 * i)
            if kind != 4:  # PT_NOTE
                continue
            p, end = at + off, at + off + size
            while p + 12 <= end:
                namesz, descsz, note = struct.unpack_from("<III", data, p)
                name = data[p + 12:p + 12 + namesz].rstrip(b"\0")
                desc = p + 12 + (namesz + 3) // 4 * 4
                if name == b"AMDGPU" and note == 32:
                    meta = msgpack.unpackb(data[desc:desc + descsz])
                    out.update((k[".name"], k) for k in meta["amdhsa.kernels"])
                p = desc + (descsz + 3) // 4 * 4


def test_split_hopping_terms_spill_no_registers(kq):
    """The waves of a split hopping term run code of their own behind branches on the wave index; a
    scalar register that lives across them in a spill slot is what such code was once compiled
    wrongly with, and a vector register in scratch memory would cost what the split gains."""
    from kuqcd_amd.build import LIB
    split = {n: k for n, k in _kernels(LIB).items() if "k_dslash_split" in n}
    assert len(split) > 100
    bad = {n: (k[".sgpr_spill_count"], k[".vgpr_spill_count"]) for n, k in split.items()
           if k[".sgpr_spill_count"] or k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}
    assert not bad
