"""17^3 executes around the batch where a plan leaves the plane-per-workgroup kernel: a plan raced
at 200 volumes must give the oracle's transform on both sides, and write its volumes only."""
import ctypes

import numpy as np
import pytest

import oracle


@pytest.mark.gpu
@pytest.mark.parametrize("d", [-1, 1])
@pytest.mark.parametrize("prec", [0, 1])
def test_tiny_executes_of_a_larger_plan(gpu, prec, d):
    f, h = gpu.fft3d, gpu.hip
    dt, tol, tiny = ((np.complex128, 1e-13, 32), (np.complex64, 6e-7, 48))[prec]
    cus = ctypes.c_int(0)
    assert h.lib().hipDeviceGetAttribute(ctypes.byref(cus), 63, 0) == 0   # multiprocessor count
    most = tiny * cus.value // 256
    x = oracle.make_input((17, 17, 17), 200, seed=17, dist="uniform", dtype=dt)
    ref = oracle.fftn_numpy(x, sign=d) / 4913
    plan = f.Plan((17, 17, 17), 200, d, prec, f.NORMALIZE)
    plane = f.Plan((17, 17, 17), 200, d, prec, f.NORMALIZE,
                   kernel="plane_17x17x17_%s_%s_v1t320" % (("c128", "c64")[prec], "fwd" if d < 0 else "bwd"))
    din, dout = h.DeviceBuffer(x.nbytes), h.DeviceBuffer(x.nbytes)
    try:
        din.upload(x)
        for b in sorted({1, 7, 8, 9, most, most + 1, 200}):
            for p in (plan, plane):
                print(p.kernel, b, flush=True)
                dout.upload(np.full(x.shape, -7, dtype=dt))
                p.execute(din.addr, dout.addr, batch=b)
                h.synchronize()
                y = dout.download(dt, x.shape)
                assert oracle.rel_l2(y[:b], ref[:b]) <= tol, b
                assert np.all(y[b:] == -7), f"x {b}: wrote past its batch"
                if p is plan:
                    first = y
                elif b <= most:     # the same kernel, so the same bits
                    assert np.array_equal(first.view(np.uint8), y.view(np.uint8)), b
    finally:
        plan.close()
        plane.close()
        din.close()
        dout.close()
