"""Mixed launches of the small-block presets ("t192", "t192_lin", "t320_lin", "t384_lin"), whose
kernel without 17^3 is another one than with it: ragged blocks of every geometry, both
directions, with 17^3, without, and with an empty 17^3 item, against the oracle -- on the host
emulator (each kernel's own LDS size, guards checked) and on the device."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMU = os.path.join(ROOT, "tests", "emu")
NAMES = ["multi_c128_t192", "multi_c128_t192_lin", "multi_c64_t320_lin", "multi_c64_t384_lin"]
SMALL = [((6, 6, 6), 23, -1), ((8, 8, 8), 7, 1), ((12, 12, 12), 3, -1), ((8, 8, 16), 4, 1),
         ((6, 6, 6), 1, 1)]
MIXES = [SMALL, SMALL + [((17, 17, 17), 0, 1)], SMALL + [((17, 17, 17), 2, 1)]]


def _inputs(name, mix):
    prec = 0 if "_c128_" in name else 1
    dt, tol = ((np.complex128, 1e-13), (np.complex64, 2e-6))[prec]
    return prec, tol, [oracle.make_input(s, max(b, 1), seed=k, dtype=dt)[:b]
                       for k, (s, b, _) in enumerate(mix)]


@pytest.mark.parametrize("mix", MIXES)
@pytest.mark.parametrize("name", NAMES)
def test_on_the_emulator(name, mix):
    subprocess.run(["make", "-s", "-C", EMU, "libfft3d_emu.so"], check=True)
    lib = ctypes.CDLL(os.path.join(EMU, "libfft3d_emu.so"))
    _, tol, xs = _inputs(name, mix)
    n = len(mix)
    ys = [np.full_like(x, np.nan) for x in xs]
    rc = lib.emu_multi(name.encode(), n, (ctypes.c_int * (3 * n))(*[v for s, _, _ in mix for v in s]),
                       (ctypes.c_int * n)(*[b for _, b, _ in mix]),
                       (ctypes.c_int * n)(*[d for _, _, d in mix]), (ctypes.c_double * n)(*[0.5] * n),
                       (ctypes.c_void_p * n)(*[x.ctypes.data for x in xs]),
                       (ctypes.c_void_p * n)(*[y.ctypes.data for y in ys]))
    assert rc == 0
    for x, y, (s, b, d) in zip(xs, ys, mix):
        assert b == 0 or oracle.rel_l2(y, 0.5 * oracle.fftn_numpy(x, sign=d)) <= tol, (s, d)


@pytest.mark.gpu
@pytest.mark.parametrize("times", [1, 60, 900])   # one block a workgroup, and claimed ones
@pytest.mark.parametrize("mix", MIXES)
@pytest.mark.parametrize("name", NAMES)
def test_on_the_device(gpu, monkeypatch, name, mix, times):
    monkeypatch.setenv("FFT3D_MX_MULTI_KERNEL", name)
    mix = [(s, b * times if s != (17, 17, 17) else b, d) for s, b, d in mix]
    prec, tol, xs = _inputs(name, mix)
    print(name, mix, flush=True)
    m = gpu.fft3d.MultiPlan(mix, precision=prec)
    try:
        assert m.info()[0] == name
        for x, y, (s, b, d) in zip(xs, m.run(xs), mix):
            assert b == 0 or oracle.rel_l2(y, oracle.fftn_numpy(x, sign=d)) <= tol, (s, d)
    finally:
        m.close()
