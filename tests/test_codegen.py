"""The device code of the superblock matvec under LLVM's machine verifier (hipcc, no GPU)."""
import os
import subprocess

import pytest

from chatokf_amd import build

SRC = """#include "okf_common.h"
#include "okf_decode.h"
#include "okf_gemv.h"
#include "okf_gemv_sb.h"
namespace okf {
#define SB(F, T, SR, P) \\
    template __global__ void gemv_sb_kernel<F, 1, 1, T, SR, false, P>(GemvGroup, uint64_t, uint32_t, uint32_t, const u32x4 *);
%s}
"""


# hipcc 7.2's si-form-memory-clauses pass loses the live range of one half of a
# two-dword load (IQ4_XS's superblock tail) where it is read as part of a vector,
# and the register is then given to an address.  sb_split keeps its dwords out
# of the vectors; the verifier, which names such a use, shows whether that holds
# (without sb_split's asm it stops at "No live subrange at use").
@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")
@pytest.mark.parametrize("fmt", ["IQ4_XS", "Q5_K", "Q4_0", "IQ4_NL", "Q8_0"])
def test_superblock_matvec_verifies(tmp_path, fmt):
    src = tmp_path / "sb.hip"
    src.write_text(SRC % "".join(f"SB({fmt}, {t}, {sr}, {p})\n" for t in (256, 512) for sr in (1, 2, 3, 5)
                                 for p in ("false", "true")))
    r = subprocess.run([build.HIPCC, *build.FLAGS, "-I", build.CSRC, "--offload-device-only", "-S", str(src), "-o",
                        str(tmp_path / "sb.s"), "-mllvm", "-verify-machineinstrs"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
