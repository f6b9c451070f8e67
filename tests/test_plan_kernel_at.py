"""fft3d_mx_plan_kernel_at: what an execute of a given batch launches, over a plan's classes."""
import numpy as np
import pytest

import oracle


def test_rejects_a_null_plan(pkg):
    lib = pkg.fft3d.load()
    lib.fft3d_mx_clear_error()
    assert lib.fft3d_mx_plan_kernel_at(None, 1) is None
    assert "kernel_at" in pkg.fft3d.last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("shape,batch", [((17, 17, 17), 200), ((24, 24, 24), 64), ((8, 8, 8), 9)])
def test_names_what_an_execute_runs(gpu, shape, batch):
    """Each execute gives the bits of a plan forced to the kernel that is reported for it."""
    f = gpu.fft3d
    x = oracle.make_input(shape, batch, seed=31)
    plan = f.Plan(shape, batch)
    assert plan.kernel_at(batch) == plan.kernel
    for b in (1, batch // 8, batch // 2, batch):
        name = plan.kernel_at(b)
        print(shape, b, name, flush=True)
        forced = f.Plan(shape, b, kernel=name)
        assert forced.kernel_at(b) == name
        y, z = plan.run(x[:b]), forced.run(x[:b])
        forced.close()
        assert np.array_equal(y.view(np.uint8), z.view(np.uint8)), (b, name)
    for b in (0, -1, batch + 1):
        with pytest.raises(ValueError):
            plan.kernel_at(b)
    plan.close()
