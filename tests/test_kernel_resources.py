"""Registers of the built kernels, from the code objects' own metadata (no GPU): a
kernel that keeps part of its state in scratch memory loses far more than the register
it saves, so none may do so unnoticed."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "llnl-spheral_amd", "lib", "libsphgpu.so")
LLVM = "/opt/rocm/llvm/bin"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"

# The 3-D mixed pair kernel that leaves the dt vote's row maxima: held to three
# wavefronts per SIMD, which two spilled registers buy (hydro.hip).
SPILLS = r"k_derivs_isoIfLi3ELb[01]ELb0ELi256ELi1ELb1EE"       # <float, 3, table, false, 256, 1, true>


def kernels(tmp_path):
    """(name as linked, metadata) of every kernel of the library."""
    fat = str(tmp_path / "fatbin")
    subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", LIB, str(tmp_path / "copy")],
                   check=True, timeout=120)
    data = open(fat, "rb").read()
    out = []
    for start in (m.start() for m in re.finditer(re.escape(MAGIC), data)):
        pos = start + len(MAGIC)
        (count,) = struct.unpack_from("<Q", data, pos)
        pos += 8
        for _ in range(count):
            offset, size, idlen = struct.unpack_from("<QQQ", data, pos)
            pos += 24
            target = data[pos:pos + idlen].decode()
            pos += idlen
            if "gfx" not in target or size == 0:
                continue
            elf = str(tmp_path / "code.o")
            with open(elf, "wb") as f:
                f.write(data[start + offset:start + offset + size])
            notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", elf], capture_output=True, text=True, check=True,
                                   timeout=120).stdout
            for block in notes.split("  - .agpr_count:")[1:]:
                meta = dict(re.findall(r"^ +\.(\w+): +(\S+)$", block, re.M))
                out.append((re.findall(r"^ +\.name: +(_Z\S+)$", block, re.M)[-1], meta))
    return out


@pytest.mark.skipif(not os.path.exists(LIB), reason="the library is not built")
@pytest.mark.parametrize("part", ["k_derivs", ""], ids=["pair kernels", "all"])
def test_no_kernel_spills_registers(tmp_path, part):
    found = kernels(tmp_path)
    assert len(found) > 100
    bad = [(n, m["vgpr_spill_count"]) for n, m in found
           if part in n and int(m["vgpr_spill_count"]) > 0 and not re.search(SPILLS, n)]
    assert not bad, bad
