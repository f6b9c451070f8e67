"""GPU: presets of the mixed launch with a second compiled kernel for launches without 17^3 items
give an item the same bits with either, alone and inside the mix."""
import numpy as np
import pytest

import oracle

SMALL = [((6, 6, 6), 23, -1), ((8, 8, 8), 13, 1), ((12, 12, 12), 5, -1), ((8, 8, 16), 7, 1)]
WITH17 = SMALL + [((17, 17, 17), 3, -1)]


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["multi_c128_t192", "multi_c128_t192_lin", "multi_c64_t320_lin",
                                  "multi_c64_t384_lin"])
def test_alone_equals_mixed(gpu, name, monkeypatch):
    f = gpu.fft3d
    prec = 0 if "_c128_" in name else 1
    dt, tol = ((np.complex128, 1e-13), (np.complex64, 2e-6))[prec]
    monkeypatch.setenv("FFT3D_MX_MULTI_KERNEL", name)
    xs = [oracle.make_input(s, b, seed=70 + k, dtype=dt) for k, (s, b, _) in enumerate(WITH17)]

    def run(items, data):
        m = f.MultiPlan(items, precision=prec)
        assert m.info()[0] == name
        print(name, items, flush=True)
        ys = m.run(data)
        m.close()
        return ys
    mixed, small = run(WITH17, xs), run(SMALL, xs[:4])
    for k, (shape, b, d) in enumerate(WITH17):
        assert oracle.rel_l2(mixed[k], oracle.fftn_numpy(xs[k], sign=d)) <= tol, (shape, d)
        alone = run([WITH17[k]], [xs[k]])[0]
        assert np.array_equal(alone.view(np.uint8), mixed[k].view(np.uint8)), shape
        if k < 4:
            assert np.array_equal(small[k].view(np.uint8), mixed[k].view(np.uint8)), shape
