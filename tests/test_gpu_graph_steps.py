"""Steps replayed from captured graphs, one and four at a time: every split of a run gives the bits of
eager stages, over several replays with other work between, after a change of dt and after a
re-layout of the operator set."""
import numpy as np
import pytest

import rbffd_gpu_amd as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("F,storage", [(1, R.F64), (3, R.F32)])
def test_replayed_steps(ctx, F, storage):
    print(f"case: replayed steps F={F} storage={storage}", flush=True)
    rng = np.random.default_rng(3)
    N, n = 700, 27
    idx = rng.integers(0, N, (N, n)).astype(np.int32)
    ws = [rng.standard_normal((N, n)) for _ in range(3)]
    u = rng.standard_normal((N, F))
    ft = R.F64 if storage == R.F64 else R.F32
    ell = R.EllOperators(ctx, idx, ws, storage=storage)
    replayed = R.RK4(ctx, ell, F, field_storage=ft, accum=R.F64)
    eager = R.RK4(ctx, ell, F, field_storage=ft, accum=R.F64, use_graph=False)
    for rk in (replayed, eager):
        rk.set_state(u)
    for dt, split in ((1e-3, (4,)), (1e-3, (1, 3, 5, 8, 0, 2)), (5e-4, (9, 4)), (5e-4, (7,))):
        for k in split:
            replayed.step(dt, k)
            eager.step(dt, k)
            assert np.array_equal(replayed.get_state(), eager.get_state()), (dt, k)
        ell.set_row_order(rng.permutation(N).astype(np.int32))
    for x in (replayed, eager, ell):
        x.close()
