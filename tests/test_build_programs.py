"""build() fills the code-object cache with the programs of the tests and the benchmark.  It builds a
library, so it needs neither pytest nor any test module, and a missing helper costs one cache entry."""
import subprocess
import sys
from pathlib import Path

REPO = Path(__file__).resolve().parent.parent

BLOCK = """
import sys
class Block:
    def find_spec(self, name, path=None, target=None):
        if name in BLOCKED or name.startswith("test_"):
            raise ModuleNotFoundError("blocked: " + name)
sys.meta_path.insert(0, Block())
sys.path.insert(0, REPO)
import __graft_entry__ as g
"""


def _run(blocked, code):
    src = f"BLOCKED, REPO = {blocked!r}, {str(REPO)!r}\n" + BLOCK + code
    r = subprocess.run([sys.executable, "-c", src], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    return r.stdout.split()


def test_definitions_need_no_test_module():
    code = """
for name, _ in g.PROGRAMS:
    if name.startswith("poly_") or name == "cert_quotient":
        continue  # from tests/systems.py, as below
    if name.startswith("cert_"):
        g._cert_system(name)
    elif name not in ("mixed4", "mixed6", "mixed8", "mixed12"):  # parts of mixed_all
        g._homotopies(name)
    print(name)
"""
    assert "solve13" in _run(["pytest", "oracle"], code)


def test_missing_helper_is_reported():
    code = """
for item in (("cyclic7", 0), ("cert_simple1", 0), ("cert_quotient", 0), ("poly_f_affine", 0)):
    assert isinstance(g._compile(item)[2], str)
print(len(g._homotopies("solve9")))
"""
    assert _run(["pytest", "oracle", "systems"], code) == ["1"]
