"""Register budgets that the kernels' occupancy rests on, read from the code objects
of the built library (MI355X: 512 registers per SIMD lane, so 256 leave 2 waves, 128
leave 4)."""
import os
import re
import struct
import subprocess

import pytest

from tuvok_amd import _abi

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{demangled kernel: (registers, spilled registers)} of libtvkhip.so"""
    data = open(_abi.LIB_PATH, "rb").read()
    out = {}
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        p = at + len(magic)
        n = struct.unpack_from("<Q", data, p)[0]
        p += 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" not in name or size == 0:
                continue
            elf = tmp_path_factory.mktemp("co") / "code.o"
            elf.write_bytes(data[at + off:at + off + size])
            txt = subprocess.run([READELF, "--notes", str(elf)], capture_output=True, text=True, check=True).stdout
            for k in txt.split("- .agpr_count:")[1:]:
                get = {f: re.search(r"\.%s:\s*(\S+)" % f, k).group(1) for f in ("name", "vgpr_count", "vgpr_spill_count")}
                sym = subprocess.run(["c++filt", get["name"]], capture_output=True, text=True, check=True).stdout
                sym = re.sub(r"^void |\(.*$|tvk::|\(anonymous namespace\)::", "", sym.replace("(anonymous namespace)::", "").strip())
                out[sym] = (int(get["vgpr_count"]), int(get["vgpr_spill_count"]))
        at = data.find(magic, at + 1)
    return out


@pytest.mark.skipif(not (os.path.exists(READELF) and os.path.exists(_abi.LIB_PATH)), reason="needs the built library")
def test_traversal_keeps_two_waves(kernels):
    leap = {k: v for k, v in kernels.items() if k.startswith("leap_kernel<")}
    assert len(leap) == 12
    for k, (regs, spill) in leap.items():
        # the form for frames of few tiles, which do not fill two waves, may take more
        few = k == "leap_kernel<0, true, unsigned short, true>"
        assert regs <= (264 if few else 256) and spill == 0, (k, regs, spill)


@pytest.mark.skipif(not (os.path.exists(READELF) and os.path.exists(_abi.LIB_PATH)), reason="needs the built library")
@pytest.mark.parametrize("pattern,count,regs,spill", [
    (r"march_kernel<1, \w+, unsigned \w+, false, 0>", 4, 128, 0),    # 2D
    (r"march_kernel<1, \w+, unsigned \w+, true, 0>", 4, 128, 4),
    (r"march_kernel<2, false, unsigned \w+, \w+, 0>", 4, 128, 8),    # isosurface
    (r"march_kernel<0, false, unsigned \w+, \w+, 0>", 4, 128, 0),    # 1D unlit, lit
    (r"march_kernel<0, true, unsigned \w+, \w+, 0>", 4, 168, 0),
    (r"march_kernel_learn<", 16, 168, 16),
    (r"batch_kernel<\d, \w+, unsigned \w+, \w+, 0>", 20, 128, 2),
    (r"batch_kernel<\d, \w+, unsigned \w+, \w+, 1>", 16, 168, 16)])
def test_march_budgets(kernels, pattern, count, regs, spill):
    """4 waves where 128 registers are named, 3 where 168 are, and the spills that the
    comments beside the kernels state."""
    found = {k: v for k, v in kernels.items() if re.match(pattern, k)}
    assert len(found) == count
    for k, v in found.items():
        assert v[0] <= regs and v[1] <= spill, (k, v)
