"""CPU check of the built gfx950 code: registers of kernels whose speed hangs
on the waves that fit a SIMD (512 registers, handed out in eights)."""
import os
import re
import subprocess

import test_isa_hazards as H


def _registers(tmp_path):
    """vgpr_count of every kernel of the library, by mangled name."""
    H._disassemble(tmp_path)  # leaves the code objects b<k>.o behind
    regs = {}
    for f in sorted(tmp_path.glob("b*.o")):
        notes = subprocess.run([os.path.join(H.LLVM, "llvm-readelf"), "--notes", str(f)], check=True,
                               capture_output=True, text=True).stdout
        for k in re.split(r"\n\s+- \.agpr_count", notes)[1:]:
            name = re.search(r"\.name:\s+(\S+)", k).group(1)
            regs[name] = int(re.search(r"\.vgpr_count:\s+(\d+)", k).group(1))
    return regs


def test_single_shamir_force_keeps_four_waves(tmp_path):
    """The Shamir force of one (R, X2) pair is bound by loads in flight: at 128
    registers or fewer four waves fit a SIMD (32^3 x 64: 73 us, with three 75)."""
    regs = {n: v for n, v in _registers(tmp_path).items() if "k_derivs_segILi0E" in n}
    assert len(regs) == 1, regs
    assert max(regs.values()) <= 128, regs
