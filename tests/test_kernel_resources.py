"""Register spills of the built kernels, from the metadata of the library's own
code object: a kernel with a private segment makes the runtime allocate scratch
memory when it is first launched, which the zero-allocation solve may not."""
import os
import re
import struct

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
NT_AMDGPU_METADATA = 32


def _code_objects(so):
    """The gfx950 ELFs bundled in a shared library."""
    at = so.find(MAGIC)
    while at >= 0:
        p = at + len(MAGIC)
        (count,) = struct.unpack_from("<Q", so, p)
        p += 8
        for _ in range(count):
            off, size, length = struct.unpack_from("<QQQ", so, p)
            name = so[p + 24:p + 24 + length]
            p += 24 + length
            if b"gfx950" in name and size:
                yield so[at + off:at + off + size]
        at = so.find(MAGIC, p)


def _metadata(elf):
    """The AMDGPU metadata note (msgpack) of a code object."""
    msgpack = pytest.importorskip("msgpack")
    (shoff,) = struct.unpack_from("<Q", elf, 0x28)
    entsize, count = struct.unpack_from("<HH", elf, 0x3A)
    for k in range(count):
        kind, _, _, off, size = struct.unpack_from("<IQQQQ", elf, shoff + k * entsize + 4)
        if kind != 7:  # SHT_NOTE
            continue
        p, end = off, off + size
        while p < end:
            nlen, dlen, note = struct.unpack_from("<III", elf, p)
            d = p + 12 + (nlen + 3) // 4 * 4
            if note == NT_AMDGPU_METADATA:
                return msgpack.unpackb(elf[d:d + dlen], raw=False)
            p = d + (dlen + 3) // 4 * 4
    return None


@pytest.fixture(scope="module")
def kernels(ox):
    from ogs5_amd import _lib
    with open(_lib.LIB_PATH, "rb") as f:
        so = f.read()
    found = {}
    for elf in _code_objects(so):
        for k in (_metadata(elf) or {}).get("amdhsa.kernels", []):
            found[k[".name"]] = k
    assert found
    return found


# (mangled: template arguments <double, ...>, and the FP64-only kernels)
NO_ALLOC = [r"k_cg_residentId", r"k_bi_residentId", r"k_cg_oneI", r"k_bi_oneI", r"k_diag_crs",
            r"k_noalloc_setup", r"k_(cg|bi)_\w*I(Li9E)?dd?", r"k_(cg|bi)_init_final"]


@pytest.mark.parametrize("pattern", NO_ALLOC)
def test_zero_allocation_kernels_need_no_scratch(kernels, pattern):
    names = [n for n in kernels if re.search(pattern, n)]
    assert names
    spilled = {n: kernels[n][".private_segment_fixed_size"] for n in names
               if kernels[n][".private_segment_fixed_size"]}
    assert not spilled
