"""A stepper whose dt changes with every call pays for no captured graph: its calls take the time of calls
with one dt (they took 1.5 times as long), and they give the bits of eager steps."""
import time

import numpy as np
import pytest

import rbffd_gpu_amd as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [1, 4, 6])
def test_changing_dt(ctx, steps):
    print(f"case: changing dt, {steps} steps a call", flush=True)
    rng = np.random.default_rng(steps)
    N, n = 4096, 31
    idx = ((np.arange(N)[:, None] + rng.integers(0, 60, (N, n))) % N).astype(np.int32)
    ell = R.EllOperators(ctx, idx, [rng.standard_normal((N, n)) for _ in range(3)])
    u = rng.standard_normal(N)
    one, new, eager = (R.RK4(ctx, ell, 1, use_graph=g) for g in (True, True, False))
    for rk in (one, new, eager):
        rk.set_state(u)
    t_one, t_new = [], []
    for i in range(80):
        for rk, dt, t in ((one, 1e-6, t_one), (new, 1e-6 * (1.0 + 1e-3 * i), t_new)):
            ctx.sync()
            t0 = time.perf_counter()
            rk.step(dt, steps)
            ctx.sync()
            t.append(time.perf_counter() - t0)
        eager.step(1e-6 * (1.0 + 1e-3 * i), steps)
    assert np.array_equal(new.get_state(), eager.get_state())
    assert np.median(t_new[10:]) < 1.25 * np.median(t_one[10:]), (np.median(t_new), np.median(t_one))
    for x in (one, new, eager, ell):
        x.close()
