"""Kernels that store 16 bytes a lane ("...l") with complex64 buffers that are aligned to one
element only, at batches that end inside a block: the oracle's transform, and not a byte beside
the batch."""
import numpy as np
import pytest

import oracle


@pytest.mark.gpu
@pytest.mark.parametrize("name,batches", [
    ("fused_6x6x6_c64_{}_v4t144l", (1, 4, 5, 403)), ("fused_6x6x6_c64_{}_v8t288l", (3, 9)),
    ("fused_6x6x6_c128_{}_v4t144l", (1, 5, 403)),
    ("pipe_17x17x17_c64_{}_v1t320p4_foldl", (1, 2, 1500)),
    ("xres_24x24x24_c64_{}_v1r1t192h8l", (1, 9)), ("xres_36x36x36_c64_{}_v1r1t448h12l", (1, 3)),
    ("xres_36x36x36_c64_{}_v1r2t256h6l", (2,)), ("xres_36x36x36_c64_{}_v1r2t448h9l", (2,))])
@pytest.mark.parametrize("d", [-1, 1])
def test_wide_stores_at_element_alignment(gpu, name, batches, d):
    f, h = gpu.fft3d, gpu.hip
    name = name.format("fwd" if d < 0 else "bwd")
    shape = tuple(int(n) for n in name.split("_")[1].split("x"))
    prec = 0 if "_c128_" in name else 1
    dt, tol = ((np.complex128, 1e-13), (np.complex64, 6e-7))[prec]
    V = shape[0] * shape[1] * shape[2]
    for b in batches:
        x = oracle.make_input(shape, b, seed=b, dist="uniform", dtype=dt)
        for off in (1, 2, 15):     # elements past a 256-byte boundary
            size = (off + b * V + 32) * x.itemsize
            din, dout = h.DeviceBuffer(size), h.DeviceBuffer(size)
            plan = f.Plan(shape, b, d, prec, kernel=name)
            try:
                host = np.full(size // x.itemsize, -7, dtype=dt)
                dout.upload(host)
                host[off:off + b * V] = x.ravel()
                din.upload(host)
                print(name, b, off, flush=True)
                plan.execute(din.addr + off * x.itemsize, dout.addr + off * x.itemsize)
                h.synchronize()
                y = dout.download(dt, host.shape)
                got = y[off:off + b * V].reshape(x.shape)
                assert oracle.rel_l2(got, oracle.fftn_numpy(x, sign=d)) <= tol
                assert np.all(y[:off] == -7) and np.all(y[off + b * V:] == -7), "wrote beside its batch"
            finally:
                plan.close()
                din.close()
                dout.close()
