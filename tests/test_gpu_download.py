"""Reading fields back: the copies go through pinned slots of 1 MiB and, from
8 MiB on, several threads; a call that finds the slots held by another
thread's, or whose buffer the caller pinned, copies directly.  Bytes must be those uploaded, whatever the path."""
import ctypes
import subprocess
import sys
import threading
from pathlib import Path

import numpy as np
import pytest

from goferro import FIELD_M, Context, Problem, workloads

pytestmark = pytest.mark.gpu


def film(n, seed):
    prob = Problem(shape=(1, 1, n), spacing=(2e-9, 2e-9, 2e-9), materials=[workloads.yig_material()],
                   material_cell=np.ones((1, 1, n), np.uint32), dt=1e-14, periodic=(True, True, True))
    return prob, np.random.default_rng(seed).standard_normal((3, 1, 1, n))


# one double; a field of just one slot and one cell more; a component of
# exactly one slot and one more and one fewer double; the field just below, at and above the threads' threshold; many
# slots with an odd tail
@pytest.mark.parametrize("n", [1, 43690, 43691, 131071, 131072, 131073, 349525, 349526, 1400011])
def test_field_comes_back_whole(n):
    print("case download", n, file=sys.stderr, flush=True)
    prob, m = film(n, n)
    c = Context(prob)
    c.upload(FIELD_M, m)
    np.testing.assert_array_equal(c.download(FIELD_M), m)
    want = m.reshape(3, -1).sum(axis=1) / n
    np.testing.assert_allclose(c.average(), want, rtol=0, atol=n * 2.0**-53 * np.abs(m).mean() * 4)
    c.close()


@pytest.mark.parametrize("n", [1, 43690, 43691, 131072, 349525, 349526, 1400011])
def test_field_comes_back_whole_each_time(n):
    """The read-backs before the slots are there, the one that allocates them
    and those after it."""
    print("case repeated download", n, file=sys.stderr, flush=True)
    prob, m = film(n, n + 1)
    c = Context(prob)
    c.upload(FIELD_M, m)
    for _ in range(6 if n <= 43690 else 3 + 16 * 4 * 2**20 // (24 * n)):
        np.testing.assert_array_equal(c.download(FIELD_M), m)
    c.close()


def test_threads_read_their_own_contexts():
    print("case download from threads", file=sys.stderr, flush=True)
    sizes = [1000, 140000, 400000, 900000]
    ctxs = []
    for i, n in enumerate(sizes):
        prob, m = film(n, 50 + i)
        c = Context(prob)
        c.upload(FIELD_M, m)
        ctxs.append((c, m))
    bad = []
    together = threading.Barrier(len(ctxs))

    def read(c, m):
        for _ in range(12):
            together.wait(timeout=60)
            if not np.array_equal(c.download(FIELD_M), m):
                bad.append(m.shape)

    threads = [threading.Thread(target=read, args=x) for x in ctxs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for c, _ in ctxs:
        c.close()
    assert not bad


@pytest.mark.parametrize("n", [1, 43691, 349526, 1400011])
def test_pinned_buffer_comes_back_whole(n):
    """A buffer from the HIP runtime the library links, by its own allocator."""
    print("case pinned download", n, file=sys.stderr, flush=True)
    prob, m = film(n, n)
    c = Context(prob)
    c.upload(FIELD_M, m)
    hip = ctypes.CDLL("libamdhip64.so.7")
    ptr = ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(ptr), ctypes.c_size_t(24 * n), ctypes.c_uint(0)) == 0
    out = ctypes.cast(ptr, ctypes.POINTER(ctypes.c_double))
    assert c.lib.gf_download(c._h, FIELD_M, out, 3 * n) == 0
    np.testing.assert_array_equal(np.ctypeslib.as_array(out, (3 * n,)), m.ravel())
    assert hip.hipHostFree(ptr) == 0
    c.close()


NO_PINNED = """
#include <stddef.h>
int hipHostMalloc(void** p, size_t n, unsigned flags) { (void)p; (void)n; (void)flags; return 2; }
"""

CHILD = """
import ctypes, sys
sys.path.insert(0, sys.argv[2])
ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)   # before the library: its hipHostMalloc is this one
import numpy as np
from goferro import FIELD_M, Context, Problem, workloads
for n in (1000, 400000):
    prob = Problem(shape=(1, 1, n), spacing=(2e-9,) * 3, materials=[workloads.yig_material()],
                   material_cell=np.ones((1, 1, n), np.uint32), dt=1e-14, periodic=(True,) * 3)
    m = np.random.default_rng(n).standard_normal((3, 1, 1, n))
    c = Context(prob)
    c.upload(FIELD_M, m)
    want = m.reshape(3, -1).sum(axis=1) / n
    for _ in range(20):
        assert np.array_equal(c.download(FIELD_M), m)
        np.testing.assert_allclose(c.average(), want, rtol=0, atol=n * 2.0**-53 * np.abs(m).mean() * 4)
    c.step(1)   # no error left for the next launch
    c.close()
print("no pinned memory: whole")
"""


def test_without_pinned_memory(tmp_path):
    """A process whose pinned allocations all fail (hipErrorOutOfMemory) reads
    fields and averages all the same."""
    print("case no pinned memory", file=sys.stderr, flush=True)
    (tmp_path / "nopin.c").write_text(NO_PINNED)
    lib = tmp_path / "libnopin.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(tmp_path / "nopin.c")], check=True)
    root = Path(__file__).resolve().parent.parent / "go-ferro_amd"
    out = subprocess.run([sys.executable, "-c", CHILD, str(lib), str(root)], capture_output=True, text=True, timeout=90)
    assert out.returncode == 0 and "whole" in out.stdout, out.stdout + out.stderr


def test_average_recurs():
    """The averages with copied sums and, from the fourth on, with sums written
    to pinned memory: the same to the last bit."""
    print("case recurring average", file=sys.stderr, flush=True)
    for n in (1, 255, 70001, 400000):
        prob, m = film(n, n)
        c = Context(prob)
        c.upload(FIELD_M, m)
        first = c.average()
        for _ in range(12):
            np.testing.assert_array_equal(c.average(), first)
        c.upload(FIELD_M, -m)
        np.testing.assert_array_equal(c.average(), -first)
        c.close()
