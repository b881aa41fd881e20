"""The read-back of fields (gf_hostio.hip) on the host, over a HIP runtime of
the driver's own in which every call can fail (tests/cpp/hostio_driver.hip)."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    from goferro import _build
    exe = tmp_path_factory.mktemp("hostio") / "hostio_driver"
    subprocess.run([_build.hipcc(), "--offload-host-only", "-std=c++17", "-O1", "-pthread",
                    str(ROOT / "tests" / "cpp" / "hostio_driver.hip"), "-o", str(exe)], check=True)
    return exe


@pytest.mark.parametrize("case", ["whole", "pays", "sums", "known", "unavailable", "errors", "host_limits", "contended"])
def test_read_back(driver, case):
    """whole: every byte, read only after it was waited for, from contexts of
    the caller's current device and of another; the slots given back with the
    last context.  pays: no slot is allocated before it saves what it costs.
    sums: the same of an average's pinned sums.  known: memory the caller pinned is copied to directly.
    unavailable: no slot to be had is a direct copy, no event a wait for the
    stream.
    errors: a copy, record or wait that fails is the call's error.  host_limits:
    allocations or threads that fail are no exception.  contended: another
    thread's slots are not waited for."""
    out = subprocess.run([str(driver), case], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stdout + out.stderr
