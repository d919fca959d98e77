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
    assert len(leap) == 10
    for k, (regs, spill) in leap.items():
        assert regs <= 256 and spill == 0, (k, regs, spill)
