"""Reading fields back: the copies go through pinned slots of 1 MiB and, from
8 MiB on, several threads; a call that finds the slots held by another
thread's, or whose buffer the caller pinned, copies directly.  Bytes must be those uploaded, whatever the path."""
import ctypes
import sys
import threading

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

    def read(c, m):
        for _ in range(5):
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
