"""The pair terms shared by the wave-per-item and block-per-item kernels leave
no fused multiply-add to the compiler's choice.

Both forms are to give the same bits, which holds only if every product that is
fused into a sum is fused in both.  The LLVM IR before any optimisation shows
what the source allows: an operation that may be contracted carries a flag.
"""
import os
import re
import subprocess

import pytest

from origami_amd import build as B

PAIR_TERMS = ("descreen_h", "descreen_tile_far", "tile_coef", "strip_coef")


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="needs hipcc")
@pytest.mark.parametrize("source", ["pair_kernels.hip", "pair_wide.hip"])
def test_pair_terms_spell_out_their_fused_operations(source):
    ir = subprocess.run([B.HIPCC, "-x", "hip", "--cuda-device-only", "-S", "-emit-llvm", "-Xclang",
                         "-disable-llvm-passes", os.path.join(B.CSRC, source), "-o", "-"] + B.flags(),
                        check=True, capture_output=True, text=True).stdout
    for name in PAIR_TERMS:
        found = re.findall(r"^define [^@]*@\S*%s.*?^}" % name, ir, re.S | re.M)
        assert found, name
        ops = [line.strip() for body in found for line in body.splitlines()
               if re.search(r"= (fadd|fsub|fmul) ", line) and " contract " in line]
        assert not ops, (name, ops[:5])
