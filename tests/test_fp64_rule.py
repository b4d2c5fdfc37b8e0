"""The rule that fixes the arithmetic of a product in the FP32 precision modes
(ccq_amd/csrc/precision.h), on the CPU."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# products of CCSD (61 orbitals) and CCSDT (40) that the register-direct kernel
# computed in FP64 when each was a launch of its own, and the largest ones of
# each kind in a search over sides of 1 to 60000 and K of 1 to 30000
FP64 = [(20412, 7, 54), (49, 49, 2916), (54, 54, 2646), (7, 54, 2646), (35, 5, 2975), (5, 5, 2975), (2435, 53, 279),
        (4225, 28, 247), (2530, 45, 287), (2339, 61, 216), (12, 60000, 10000), (64, 60000, 20), (32, 3000000, 29), (1, 1, 1)]
FP32 = [(900, 900, 900), (8100, 100, 8100), (64, 4375, 1225), (65, 65, 8), (35, 153125, 35)]


def test_rule(tmp_path):
    cases = FP64 + FP32
    src = tmp_path / "t.cpp"
    src.write_text('#include "precision.h"\n#include <cstdio>\nint main() {\n' + "".join(
        f'  std::printf("%d\\n", ccqk::fp64_in_mixed({m}, {n}, {k}));\n' for m, n, k in cases) + "}\n")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-I", os.path.join(ROOT, "ccq_amd", "csrc"), str(src),
                    "-o", str(tmp_path / "t")], check=True)
    out = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True, check=True).stdout.split()
    assert out == ["1"] * len(FP64) + ["0"] * len(FP32)
