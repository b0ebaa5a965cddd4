"""What the compiler gave the kernels of the built library: registers, spills and
scratch memory, read from the code objects' metadata.  A kernel that spills, or
takes so many registers that a wave less fits, gives the same results, only
later, so no other test notices."""
import os
import re
import struct

import pytest

msgpack = pytest.importorskip("msgpack")

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pdesolver.jl_amd")
LIB = os.path.join(PKG, "pdes_amd", "libpdes_amd.so")
# registers of a lane at which n waves fit a SIMD (512 registers, in steps of 8)
REGS_AT_WAVES = {3: 168, 4: 128}


def _code_objects(data):
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        at = m.start()
        n, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            ident = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"amdgcn" in ident:
                yield data[at + off:at + off + size]


def _metadata(elf):
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        kind, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        off, size = struct.unpack_from("<QQ", elf, shoff + i * shentsize + 24)
        p = off
        while kind == 7 and p < off + size:
            namesz, descsz, typ = struct.unpack_from("<III", elf, p)
            desc = p + 12 + (namesz + 3) // 4 * 4
            if typ == 32:
                return msgpack.unpackb(elf[desc:desc + descsz], strict_map_key=False)
            p = desc + (descsz + 3) // 4 * 4
    return {}


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(LIB):
        import build_lib
        build_lib.build()
    with open(LIB, "rb") as f:
        data = f.read()
    out = {}
    for elf in _code_objects(data):
        for k in _metadata(elf).get("amdhsa.kernels", []):
            out[k[".name"]] = k
    assert out
    return out


def _matching(kernels, pattern, count):
    found = {n: k for n, k in kernels.items() if re.search(pattern, n)}
    assert len(found) == count, sorted(found)
    return found


def _no_spills(found):
    bad = {n: (k[".vgpr_spill_count"], k[".private_segment_fixed_size"]) for n, k in found.items()
           if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}
    assert not bad, bad


def test_diage_weak_form_derivatives_run_three_waves(kernels):
    """The weak form's derivative on the four diagonal-E operators."""
    found = _matching(kernels, r"euler_residual_kernelINS_7OpShapeILi2ELi\d+ELi\d+ELi\d+ELb1EEELi1E.*dualILi1E", 4)
    _no_spills(found)
    assert all(k[".vgpr_count"] <= REGS_AT_WAVES[3] for k in found.values()), \
        {n: k[".vgpr_count"] for n, k in found.items()}


def test_block_jacobi_factorizations_run_four_waves(kernels):
    """Ten operators, FP32 and FP64 blocks."""
    found = _matching(kernels, r"bjacobi_factor_kernel", 20)
    _no_spills(found)
    assert all(k[".vgpr_count"] <= REGS_AT_WAVES[4] for k in found.values()), \
        {n: k[".vgpr_count"] for n, k in found.items()}


def test_dependency_sweeps_do_not_spill(kernels):
    """The ILU(0) sweeps of ten operators, FP32 and FP64 blocks: a share of an
    element that does not stay in registers ends the loading ahead."""
    _no_spills(_matching(kernels, r"ilu_sweep_dep_kernel", 20))
