"""The certifier's code objects, compiled for gfx950 without a device."""
import os
import re
import subprocess
import sys

import pytest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
COMPILE = """
import ctypes, sys
sys.path.insert(0, {pkg!r})
from hcgpu import abi
from hcgpu.configs import parameter_product_system
from hcgpu.homotopies import _SysTapes
tapes, size = _SysTapes(parameter_product_system()), ctypes.c_size_t()
st = tapes.struct()
rc = abi.lib().hcg_certifier_compile_only(ctypes.byref(st), 3, ctypes.byref(size))
assert rc == 0, abi.lib().hcg_last_error()
"""


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_four_waves_per_simd(tmp_path):
    """Every kernel of a certifier with split tapes keeps to 128 registers a lane."""
    pkg = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "homotopycontinuation.jl_amd")
    subprocess.run([sys.executable, "-c", COMPILE.format(pkg=pkg)], check=True, env=dict(os.environ, HCGPU_CACHE_DIR=str(tmp_path)))
    (code,) = tmp_path.glob("*.co")
    notes = subprocess.run([READELF, "--notes", str(code)], capture_output=True, text=True, check=True).stdout
    regs = [int(v) for v in re.findall(r"\.vgpr_count: +(\d+)", notes)]
    assert len(regs) >= 2 and max(regs) <= 128, regs
