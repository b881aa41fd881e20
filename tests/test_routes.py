"""The size rules that pick a kernel's offset width, checked on the host
against the offsets the kernel forms (tests/cpp/route_driver.hip), at and
around the sizes where they change."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    import goferro
    from goferro import _build
    if not goferro.LIB_PATH.exists():
        pytest.skip("libgoferro.so not built (run __graft_entry__.build())")
    exe = tmp_path_factory.mktemp("routes") / "route_driver"
    subprocess.run([_build.hipcc(), "--offload-host-only", "-std=c++17", "-O1",
                    str(ROOT / "tests" / "cpp" / "route_driver.hip"), f"-L{goferro.LIB_PATH.parent}", "-lgoferro",
                    f"-Wl,-rpath,{goferro.LIB_PATH.parent}", "-o", str(exe)], check=True)
    return exe


@pytest.mark.parametrize("rule", ["elastic_force", "magnet_list", "cell_div"])
def test_offset_rule(driver, rule):
    """elastic_force: the cell arrays and, with the Liao plane, a history slot
    of 12 nx ny elements stay within 32-bit byte offsets, and no grid that
    does is refused the 32-bit form.  magnet_list: the stage over a list of FM
    cells uses 64-bit offsets from 2^28 cells on.  cell_div: the multiplications
    that stand for divisions of a cell index by an axis length are exact up to
    the largest index the 32-bit kernels take."""
    out = subprocess.run([str(driver), rule], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
