"""The Stokes set-up on the device: a stencil that names a node twice or misses its centre is refused
with the stencil's row and node, whatever the row order; the first bad position decides."""
import numpy as np
import pytest

import rbffd_gpu_amd as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("N,n", [(70, 3), (300, 31), (300, 64)])
def test_bad_stencils(ctx, N, n, reverse):
    print(f"case: stokes set-up N={N} n={n} reverse={reverse}", flush=True)
    good = ((np.arange(N)[:, None] + np.arange(n)[None, :]) % N).astype(np.int32)
    ws = [np.ones((N, n))] * 4

    def create(st):
        e = R.EllOperators(ctx, st, ws, storage=R.F64, types=[R.LSFC, R.XSFC, R.YSFC, R.ZSFC])
        if reverse:
            e.set_row_order(np.arange(N)[::-1].copy())
        try:
            R.Stokes(ctx, e).close()
        finally:
            e.close()

    create(good)
    twice, missing = good.copy(), good.copy()
    twice[5, n - 1] = twice[5, 1]
    missing[9, 0] = (9 + n) % N  # not the centre
    with pytest.raises(R.RbfxError, match=f"stencil 5 holds node {good[5, 1]} twice"):
        create(twice)
    with pytest.raises(R.RbfxError, match="stencil 9 does not contain its centre"):
        create(missing)
    both = twice.copy()
    both[9] = missing[9]
    with pytest.raises(R.RbfxError, match="stencil 9 does not" if reverse else "stencil 5 holds"):
        create(both)
