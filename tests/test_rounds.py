"""Residue-split launches by rounds ("xres_..._v1rounds"): full rounds in one form, the remainder
in another, at the batch sizes where the split changes -- against the oracle on the host
emulator, and on the device at its own round sizes against a single-form kernel."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMU = os.path.join(ROOT, "tests", "emu")


# CUs -> batches.  Volumes a round at R workgroups a volume, W a CU: 8 * (CUs / 8 * W // R); with
# 32 CUs 16 at R = 2, 8 at R = 4 and 0 above, so 19 volumes of 24x24x48 run as 16 + 3 and 25 as
# 16 + 9 > 8: all in the last form.  8 CUs hold no round of any complex128 form.
@pytest.mark.parametrize("cus,batches", [(8, (1, 9)), (32, (3, 16, 17, 19, 25)), (96, (8, 9, 17))])
@pytest.mark.parametrize("name,shape,prec", [
    ("xres_24x24x48_c128_fwd_v1rounds", (24, 24, 48), 0),
    ("xres_24x24x24_c64_bwd_v1rounds", (24, 24, 24), 1)])
def test_rounds_on_the_emulator(name, shape, prec, cus, batches):
    subprocess.run(["make", "-s", "-C", EMU, "libfft3d_emu.so"], check=True)
    lib = ctypes.CDLL(os.path.join(EMU, "libfft3d_emu.so"))
    lib.emu_transform.argtypes = [ctypes.c_char_p, ctypes.c_void_p, ctypes.c_void_p,
                                  ctypes.c_long, ctypes.c_double, ctypes.c_int]
    dt, tol = ((np.complex128, 1e-13), (np.complex64, 2e-6))[prec]
    sign = -1 if "_fwd_" in name else 1
    lib.emu_set_cus(cus)
    try:
        for b in batches:
            x = oracle.make_input(shape, b, seed=b, dist="uniform", dtype=dt)
            out = np.full((b + 1,) + shape, np.nan, dtype=dt)
            assert lib.emu_transform(name.encode(), x.ctypes.data, out.ctypes.data, b, 1.0, 0) == 0
            assert oracle.rel_l2(out[:b], oracle.fftn_numpy(x, sign=sign)) <= tol, (name, cus, b)
            assert np.all(np.isnan(out[b])), f"{name} x {b}: wrote past its batch"
    finally:
        lib.emu_set_cus(32)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,prec,single,Rs", [
    ((36, 36, 36), 0, "xres_36x36x36_c128_{}_v1r6t512o2", (12, 6, 4, 2)),
    ((24, 24, 48), 0, "xres_24x24x48_c128_{}_v1r4t384o2", (8, 4, 2)),
    ((24, 24, 24), 0, "xres_24x24x24_c128_{}_v1r3t192", (6, 4)),
    ((36, 36, 36), 1, "xres_36x36x36_c64_{}_v1r3t512", (12, 6, 3, 2, 1)),
    ((24, 24, 48), 1, "xres_24x24x48_c64_{}_v1r3t256", (6, 3, 2, 1)),
    ((24, 24, 24), 1, "fused_24x24x24_c64_{}_v1t576", (6, 3, 2))])
def test_rounds_at_the_devices_round_sizes(gpu, shape, prec, single, Rs):
    f, h = gpu.fft3d, gpu.hip
    cus = ctypes.c_int(0)
    assert h.lib().hipDeviceGetAttribute(ctypes.byref(cus), 63, 0) == 0   # multiprocessor count
    rounds = [cus.value // 8 // R * 8 for R in Rs]
    batches = sorted({b for r in rounds for b in (r, r + 1)} | {1, rounds[-1] + rounds[0] + 3})
    batches = [b for b in batches if b >= 1]
    dt, tol = ((np.complex128, 1e-13), (np.complex64, 1e-6))[prec]
    top, V = batches[-1], shape[0] * shape[1] * shape[2]
    for tag, d in (("fwd", f.FORWARD), ("bwd", f.BACKWARD)):
        x = oracle.make_input(shape, top, seed=11, dist="uniform", dtype=dt)
        din, dout = h.DeviceBuffer(x.nbytes), h.DeviceBuffer(x.nbytes)
        try:
            din.upload(x)
            ref = f.Plan(shape, top, d, prec, kernel=single.format(tag))
            ref.execute(din.addr, dout.addr)
            h.synchronize()
            want = dout.download(dt, x.shape)
            few = [0, top // 2, top - 1]
            assert oracle.rel_l2(want[few], oracle.fftn_numpy(x[few], sign=d)) <= tol
            plan = f.Plan(shape, top, d, prec,
                          kernel="xres_%dx%dx%d_%s_%s_v1rounds" % (*shape, ("c128", "c64")[prec], tag))
            for b in batches:
                print(plan.kernel, b, flush=True)
                dout.upload(np.full(x.shape, -7, dtype=dt))
                plan.execute(din.addr, dout.addr, batch=b)
                h.synchronize()
                y = dout.download(dt, x.shape)
                err = np.linalg.norm((y[:b] - want[:b]).reshape(b, V), axis=1)
                assert np.all(err <= tol * np.linalg.norm(want[:b].reshape(b, V), axis=1)), b
                assert np.all(y[b:] == -7), f"x {b}: wrote past its batch"
            ref.close()
            plan.close()
        finally:
            din.close()
            dout.close()
