"""Registers and scratch of the decode attention's variants, read from the metadata of the library built here."""
import re
import shutil
import struct
import subprocess

import pytest

from turboquant_plus_amd import _lib as L

READELF = shutil.which("llvm-readelf") or shutil.which("llvm-readelf", path="/opt/rocm/llvm/bin")
BIAS_NONE, BIAS_LIST, BIAS_DENSE, BIAS_BOTH = range(4)
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """The gfx950 ELF files in the offload bundles of a host library."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        entry = at + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", data, at + len(MAGIC))[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            triple = data[entry + 24:entry + 24 + length]
            entry += 24 + length
            if b"gfx950" in triple and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + len(MAGIC))


@pytest.fixture(scope="module")
def variants(tmp_path_factory):
    """(K format, K bits, V bits, Sparse V, shared table, sets of four heads, bias, 256 dims) -> (registers, scratch bytes)"""
    if READELF is None or shutil.which("c++filt") is None:
        pytest.skip("llvm-readelf or c++filt is missing")
    found = {}
    for i, elf in enumerate(code_objects(L.LIB_PATH)):
        path = tmp_path_factory.mktemp("co") / f"{i}.co"
        path.write_bytes(elf)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for kernel in re.split(r"^  - \.agpr_count", notes, flags=re.M)[1:]:
            field = {k: re.search(rf"^    \.{k}: +(\S+)", kernel, re.M).group(1) for k in ("name", "vgpr_count", "private_segment_fixed_size")}
            found[field["name"]] = int(field["vgpr_count"]), int(field["private_segment_fixed_size"])
    plain = subprocess.run(["c++filt"], input="\n".join(found), capture_output=True, text=True, check=True).stdout.splitlines()
    res = {}
    for name, r in zip(plain, found.values()):
        m = re.search(r"k_decode_attn<([^>]*)>", name)
        if m:
            res[tuple(v == "true" if v in ("true", "false") else int(v) for v in m.group(1).split(", "))] = r
    assert res, "no decode attention kernels found"
    return res


def of(variants, bias, **want):
    names = ("kformat", "kbits", "vbits", "sparse", "share", "sets", "bias", "d256")
    return {k: r for k, r in variants.items() if k[6] == bias and all(k[names.index(n)] == v for n, v in want.items())}


def test_every_kind_of_bias_has_a_variant(variants):
    for k in of(variants, BIAS_NONE):
        assert all((*k[:6], b, k[7]) in variants for b in (BIAS_LIST, BIAS_DENSE, BIAS_BOTH)), k


def test_dense_rows_alone_do_not_pay_for_a_list(variants):
    """No scratch (a little with 256 dims, which are held to 128 registers), and next to 8-bit rows the registers of three
    wavefronts per SIMD."""
    for k, (vgprs, scratch) in of(variants, BIAS_DENSE).items():
        assert scratch <= (12 if k[7] else 0), (k, scratch)
    eight = of(variants, BIAS_DENSE, kformat=1, sets=2, sparse=False, d256=False)
    eight = {k: r for k, r in eight.items() if k[2] != 8}
    wide = {k: r for bits in (3, 4) for k, r in of(variants, BIAS_DENSE, kformat=0, kbits=bits, vbits=8, d256=True).items()}
    assert len(eight) == 3 and len(wide) == 4
    for k, (vgprs, _) in {**eight, **wide}.items():
        assert vgprs <= 168, (k, vgprs)
