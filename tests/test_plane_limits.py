"""The plane-per-workgroup 17^3 kernel serves the batches at which it was measured the quickest
(32 volumes in complex128, 48 in complex64, on 256 CUs) and none above: not as the kernel of a
plan, not as its small-batch class, and not through a verdict recorded for a nearby batch."""
import ctypes
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _most(h, prec):
    cus = ctypes.c_int(0)
    assert h.lib().hipDeviceGetAttribute(ctypes.byref(cus), 63, 0) == 0   # multiprocessor count
    return (32, 48)[prec] * cus.value // 256


def _check(plan, most):
    plane = [b for b in range(1, plan.batch + 1) if plan.kernel_at(b).startswith("plane_")]
    assert plane == list(range(1, min(most, plan.batch) + 1)), (plan.batch, plane[-1:])
    small = plan.kernel_small
    assert small is None or (not small[0].startswith("plane_") and small[1] > most), small


# In this order: a plan at the limit, then those of its power-of-two batch class and above.
@pytest.mark.gpu
@pytest.mark.parametrize("prec", [0, 1])
def test_plane_kernel_stays_within_its_limit(gpu, prec):
    f, most = gpu.fft3d, _most(gpu.hip, prec)
    for batch in (most, most + 1, 1, 2 * most - 1, 128, 200, 256, 300, 390):
        plan = f.Plan((17, 17, 17), batch, f.FORWARD, prec)
        print(batch, plan.kernel, plan.kernel_small, flush=True)
        _check(plan, most)
        plan.close()


@pytest.mark.gpu
def test_recorded_verdict_does_not_lift_the_limit(gpu, tmp_path):
    """A wisdom file that names the plane kernel for the class of 32 to 63 volumes."""
    most = _most(gpu.hip, 0)
    first = tmp_path / "first"
    code = ("import __graft_entry__ as g, sys; f = g.load_package().fft3d\n"
            "p = f.Plan((17, 17, 17), int(sys.argv[1])); print(p.kernel_at(p.batch)); p.close()")

    def child(path, batch):
        r = subprocess.run([sys.executable, "-c", code, str(batch)], cwd=ROOT, text=True, timeout=100,
                           capture_output=True, env=dict(os.environ, FFT3D_MX_WISDOM=str(path)))
        assert r.returncode == 0, r.stderr
        return r.stdout.split()[-1]
    assert not child(first, 2 * most - 1).startswith("plane_")
    keys = [line.split()[0] for line in first.read_text().splitlines()]
    assert keys
    path = tmp_path / "wisdom"
    path.write_text("".join(f"{k} plane_17x17x17_c128_fwd_v1t320\n" for k in keys))
    assert not child(path, 2 * most - 1).startswith("plane_")
