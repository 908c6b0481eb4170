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


def _shapes(evaluate, calls):
    v = evaluate([f"{c}.{f}" for c in calls for f in ("workgroups", "per_wave")])
    return list(zip(v[::2], v[1::2]))


def test_lane_shape(evaluate):
    """On 256 CUs: one lane of each wave up to one path per CU, full waves from 64 paths per CU on; no more
    workgroups than wave slots; every path has a lane or waits in the queue of a full grid."""
    n = [0, 1, 81, 256, 257, 511, 513, 6561, 256 * 63, 256 * 63 + 1, 256 * 64, 256 * 64 + 1, 262144]
    got = _shapes(evaluate, [f"lane_shape(256, 1, 0, {p}L)" for p in n])
    assert got == [(1, 1), (1, 1), (81, 1), (256, 1), (129, 2), (256, 2), (171, 3), (253, 26), (256, 63), (253, 64), (256, 64),
                   (257, 64), (1024, 64)]
    assert _shapes(evaluate, ["lane_shape(256, 2, 0, 262144L)", "lane_shape(256, 1, 1, 262144L)", "lane_shape(256, 8, 0, 100L)"]) == [
        (2048, 64), (256, 64), (100, 1)]


def test_group_shape(evaluate):
    """Four 16-lane or two 32-lane groups per wave, four waves per workgroup, 256 CUs."""
    n = [0, 1, 5, 1024, 1025, 2049, 3073, 8192, 65536]
    assert _shapes(evaluate, [f"group_shape(256, 4, 4, 0, {p}L)" for p in n]) == [
        (1, 1), (1, 1), (2, 1), (256, 1), (129, 2), (171, 3), (193, 4), (512, 4), (512, 4)]
    n = [601, 1024, 1025, 2048, 2049, 4096, 4097, 8192]
    assert _shapes(evaluate, [f"group_shape(256, 4, 2, 0, {p}L)" for p in n]) == [
        (151, 1), (256, 1), (129, 2), (256, 2), (257, 2), (512, 2), (512, 2), (512, 2)]
    assert _shapes(evaluate, ["group_shape(256, 4, 4, 1, 65536L)"]) == [(256, 4)]
