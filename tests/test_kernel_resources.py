"""CPU: registers and private memory of this library's own kernels, from the
metadata that the compiler writes beside them.  The E -> L kernels hide memory
latency behind each other's waves: a wave fewer, or a sum that goes through
private memory, costs time at every size and shows in no result.
"""
import os
import re
import struct
import subprocess

import pytest

msgpack = pytest.importorskip("msgpack")
LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mfem_amd",
                   "libh1pa.so")


def _code_objects(blob):
    """The gfx950 ELF images of every offload bundle in the library."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = blob.find(magic)
    while at >= 0:
        n, = struct.unpack_from("<Q", blob, at + 24)
        p = at + 32
        if n < 16:
            for _ in range(n):
                off, size, idlen = struct.unpack_from("<QQQ", blob, p)
                name = blob[p + 24:p + 24 + idlen]
                p += 24 + idlen
                if b"gfx950" in name and size:
                    yield blob[at + off:at + off + size]
        at = blob.find(magic, at + 24)


def _metadata(elf):
    """The AMDGPU metadata notes (type 32) of an ELF image."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + i * shentsize)
        if kind != 7:  # SHT_NOTE
            continue
        p, end = off, off + size
        while p < end:
            nlen, dlen, ntype = struct.unpack_from("<III", elf, p)
            d = p + 12 + (nlen + 3) // 4 * 4
            if ntype == 32:
                yield msgpack.unpackb(elf[d:d + dlen], raw=False, strict_map_key=False)
            p = d + (dlen + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    """{demangled name without its arguments: metadata}"""
    if not os.path.exists(LIB):
        pytest.skip("the library is not built")
    with open(LIB, "rb") as f:
        blob = f.read()
    ks = [k for e in _code_objects(blob) for m in _metadata(e) for k in m["amdhsa.kernels"]]
    names = subprocess.run(["c++filt"], input="\n".join(k[".name"] for k in ks), text=True,
                           capture_output=True, check=True).stdout.splitlines()
    short = [re.sub(r"^void ", "", n.replace("(anonymous namespace)::", "")).split("(")[0]
             for n in names]
    return {n.replace("h1pa::kern::", ""): k for n, k in zip(short, ks)}


def _of(kernels, name):
    got = {n: k for n, k in kernels.items() if n.split("<")[0] == name}
    assert got, name
    return got


def test_scatter_rows_keeps_its_sums_in_registers(kernels):
    for name, k in _of(kernels, "k_scatter_rows").items():
        assert k[".private_segment_fixed_size"] == 0, name


@pytest.mark.parametrize("name", ["k_pcg_scatter", "k_ir_scatter", "k_ir_ru_res", "k_cheb_scatter",
                                  "k_residual", "k_small_scatter", "k_small_update",
                                  "k_small_dir", "kb_scatter", "kbm_ru_res"])
def test_solver_row_kernels_run_eight_waves(kernels, name):
    """512 registers a SIMD lane: 64 a wave for eight waves."""
    for full, k in _of(kernels, name).items():
        assert k[".vgpr_count"] <= 64 and k.get(".agpr_count", 0) == 0, full
        assert k[".private_segment_fixed_size"] == 0, full
