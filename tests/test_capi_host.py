"""Host-side behaviour of the library under a HIP runtime without a device
(tests/capi/host_driver.c): runs without a GPU."""

from __future__ import annotations

import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
LIB = ROOT / "somax_amd" / "lib" / "libsomaxhip.so"
PRECISION = {"fp32": 0, "mixed": 1, "bf16x6": 2, "fp64": 3}


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = tmp_path_factory.mktemp("capi") / "host_driver"
    cmd = ["gcc", "-O1", "-std=gnu11", f"-I{ROOT / 'include'}", str(ROOT / "tests" / "capi" / "host_driver.c"), "-o",
           str(exe), "-rdynamic", "-ldl"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr

    def run(nx, ny, nl, precision):
        args = [str(exe), str(LIB), *map(str, (nx, ny, nl, PRECISION[precision]))]
        res = subprocess.run(args, capture_output=True, text=True, timeout=60)
        assert res.returncode == 0, (res.returncode, res.stderr)
        return {k: int(v) for k, v in (line.split() for line in res.stdout.splitlines())}

    return run


@pytest.mark.parametrize("precision", sorted(PRECISION))
@pytest.mark.parametrize("n", [30, 130, 256, 512, 600])
def test_second_device_has_its_lds_limits_raised(driver, n, precision):
    """Plans on device 0 and then on device 1 of one process: every launch on device 1
    stays within the dynamic LDS limit set there."""
    out = driver(n, n, 3, precision)
    assert out["launches"] >= 14
    assert out["refused"] == 0


@pytest.mark.parametrize("precision", sorted(PRECISION))
@pytest.mark.parametrize("n", [30, 130, 512])
def test_calls_allocate_no_host_memory(driver, n, precision):
    """An inversion, a right-hand side and a step allocate nothing on the host."""
    assert driver(n, n, 3, precision)["allocations"] == 0
