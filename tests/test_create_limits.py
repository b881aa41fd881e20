"""gf_create when host memory runs out: GF_ERR_ALLOC, never an exception through
the C entry.  Every allocation of the size of a grid's cell codes fails once,
in a process of its own whose operator new counts them."""
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

COUNTING_NEW = """
#include <cstddef>
#include <cstdlib>
#include <new>
static std::size_t from = ~std::size_t{0};
static int seen = 0, fails = -1;
extern "C" void arm(std::size_t bytes, int k) { from = bytes; seen = 0; fails = k; }
extern "C" int count() { return seen; }
void* operator new(std::size_t n) {
    if (n >= from && seen++ == fails) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
"""

CHILD = """
import ctypes, sys
sys.path.insert(0, sys.argv[2])
new = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)   # before the library: its operator new is this one
import numpy as np
from goferro import Context, GoFerroError, Problem, workloads
shape = (40, 30, 20)
n = 40 * 30 * 20

def create(cell, k):
    prob = Problem(shape=shape, spacing=(2e-9,) * 3, materials=[workloads.yig_material(), workloads.yig_material()],
                   material_cell=cell, dt=1e-14, periodic=(True, True, False))
    new.arm(ctypes.c_size_t(4 * n), k)
    try:
        Context(prob).close()
        text = "created"
    except GoFerroError as e:
        text = str(e)
    seen = new.count()
    new.arm(ctypes.c_size_t(2**63), -1)
    return text, seen

one = np.ones(shape, np.uint32)
two = one.copy()
two[20:] = 2
for cell in (one, two):
    whole, seen = create(cell, -1)
    assert "failed (-4)" not in whole and seen >= 1, (whole, seen)
    for k in range(seen):
        text, _ = create(cell, k)
        assert "failed (-4)" in text and "allocation" in text, (k, text)
print("refused")
"""


def test_create_without_host_memory(tmp_path):
    import goferro
    if Path("/dev/kfd").exists():
        pytest.skip("with a GPU the allocations of the HIP runtime would count too")
    if not goferro.LIB_PATH.exists():
        pytest.skip("libgoferro.so not built (run __graft_entry__.build())")
    (tmp_path / "new.cpp").write_text(COUNTING_NEW)
    lib = tmp_path / "libnew.so"
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-o", str(lib), str(tmp_path / "new.cpp")], check=True)
    out = subprocess.run([sys.executable, "-c", CHILD, str(lib), str(ROOT / "go-ferro_amd")], capture_output=True,
                         text=True, timeout=60)
    assert out.returncode == 0 and "refused" in out.stdout, out.stdout + out.stderr
