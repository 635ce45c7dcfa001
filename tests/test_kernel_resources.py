"""What the compiler gave the kernels, from the metadata of the built library's
own code objects (llvm-readelf; no GPU)."""
import os
import re
import struct
import subprocess

import pytest

from sengapy import abi

READELF = "/opt/rocm/lib/llvm/bin/llvm-readelf"
LDS, BLK = 163840, 256   # LDS of a CU; threads of a point kernel's block

pytestmark = pytest.mark.skipif(not os.path.exists(READELF), reason="llvm-readelf not present")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: {metadata key: value}} of every kernel in the library."""
    if not os.path.exists(abi.LIBPATH):
        import build
        build.build_library()
    lib = open(abi.LIBPATH, "rb").read()
    at = [m.start() for m in re.finditer(b"\x7fELF", lib)]
    at = [p for p in at if struct.unpack_from("<H", lib, p + 18)[0] == 224]   # EM_AMDGPU
    tmp = tmp_path_factory.mktemp("code") / "object"
    out = {}
    for p, end in zip(at, at[1:] + [len(lib)]):
        tmp.write_bytes(lib[p:end])
        text = subprocess.run([READELF, "--notes", str(tmp)], capture_output=True, text=True).stdout
        for block in text.split("\n  - .")[1:]:
            name = re.search(r"^\s*\.name:\s+(_Z\w+)", block, re.M)
            if name:
                out[name.group(1)] = {k: int(v) for k, v in re.findall(r"\.(\w+):\s+(\d+)\s*$", block, re.M)}
    assert len(out) > 500
    return out


def _get(kernels, pattern):
    got = [v for k, v in kernels.items() if re.match(pattern, k)]
    assert got, pattern
    return got


@pytest.mark.parametrize("ns", range(2, 19))
def test_fill_up_rows_cost_no_block(kernels, ns):
    """The point kernels of a mechanism read at run time hold a block's
    concentrations and Gibbs functions in LDS.  What they hold beside them
    leaves as many blocks on a CU (up to the four their registers allow) as
    the NS rows alone, and exp_t's 512 bytes (the table, or the vote of
    k_rate64) in FP64."""
    for kernel, size, extra in ((rf"_ZN2sg6k_primILi{ns}ELb0E", 8, 512), (rf"_ZN2sg8k_rate64ILi{ns}ELb0E", 8, 512),
                                (rf"_ZN2sg9k_prim_mxILi{ns}ELb0E", 4, 0)):
        want = min(4, LDS // (ns * BLK * (size + 8) + extra))
        for k in _get(kernels, kernel):
            assert min(4, LDS // k["group_segment_fixed_size"]) == want, (kernel, k["group_segment_fixed_size"])


def test_cross_kernels_do_not_spill(kernels):
    """k_final<BND, NS, R, true>: every form between the substages keeps its
    three fields' derivatives in registers."""
    got = _get(kernels, r"_ZN2sg7k_finalILb[01]ELi\d+E[df]Lb1E")
    assert len(got) >= 2 * 2 * 17
    assert [k["vgpr_spill_count"] for k in got if k["vgpr_spill_count"]] == []
