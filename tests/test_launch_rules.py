"""Launch rules of the host runtime (csrc/hcg_launch_rules.h), compiled for the CPU."""
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "homotopycontinuation.jl_amd" / "csrc"


@pytest.fixture(scope="module")
def evaluate(tmp_path_factory):
    """evaluate([expression, ...]): the values of C++ expressions over the rules, as integers."""
    d = tmp_path_factory.mktemp("rules")

    def run(exprs):
        src = '#include <cstdio>\n#include "hcg_launch_rules.h"\nusing namespace hcg;\nint main() {\n'
        src += "".join(f'  std::printf("%ld\\n", (long)({e}));\n' for e in exprs) + "}\n"
        (d / "t.cpp").write_text(src)
        subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(d / "t.cpp"), "-o", str(d / "t")], check=True)
        return [int(v) for v in subprocess.run([str(d / "t")], capture_output=True, text=True, check=True).stdout.split()]

    return run


# coefficients, table, saved operations, program operations
N10 = (718, 14 * 200 + 10 * 518, 12206, 12206)  # n = 10, coefficients affine in 16 parameters
PROD3 = (63, 14 * 18 + 10 * 45, 146, 189)  # n = 3, products of parameters
TINY = (2, 24, 64, 64)
HUGE = (1, 1 << 29, 10**6, 10**6)


def test_certify_with_tables(evaluate):
    """Tables where candidates share parameter vectors or the vectors are few; never more than the budget."""
    calls = [(64, 1, N10, 1), (1, 1, N10, 1), (16000, 16, N10, 1), (262144, 256, N10, 1), (16384, 16384, N10, 1),
             (40000, 40000, N10, 0), (262144, 262144, N10, 0), (262144, 32768, N10, 1), (10**6, 67277, N10, 1),
             (2 * 10**6, 67278, N10, 0), (4096, 4096, PROD3, 1), (4372, 4372, PROD3, 1), (4373, 4373, PROD3, 0),
             (9000, 4661, PROD3, 1), (9000, 4662, PROD3, 0), (65536, 65536, PROD3, 0), (16, 1, TINY, 1),
             (17, 2, TINY, 1), (16, 2, TINY, 0), (1, 1, HUGE, 1), (2, 2, HUGE, 0)]
    args = ["{%dL, %dL, %dL, %dL}" % c[2] for c in calls]
    got = evaluate([f"certify_with_tables({c[0]}L, {c[1]}L, CertSplit{a})" for c, a in zip(calls, args)])
    assert got == [c[-1] for c in calls]
