"""The ILU(0) sweeps in FP32, as the FP32 inner solves use them, at the edges of their kernel: every variant of entries
per side (32, 40, 48, 56 and 64), chunks of one row, and values older than the ring in LDS. One GMRES step in
FP32 refinement returns a multiple of the preconditioned right-hand side, M^-1 b scaled twice in FP32:
it is compared element by element with substitutions in FP32 with the rounded factor, each sum
in column order."""
import numpy as np
import pytest

import rbffd_gpu_amd as R
from test_gpu_sweeps import stencils

pytestmark = pytest.mark.gpu


def substituted(col, F, v):
    """The two sweeps over v (N, 3) in FP32; col (N, n) ascending, F the factor's entries."""
    v, (N, n) = v.copy(), col.shape
    for r in range(N):
        s = v[r].copy()
        for q in range(np.searchsorted(col[r], r)):
            s = s - F[r, q] * v[col[r, q]]
        v[r] = s
    for r in range(N - 1, -1, -1):
        s, d = v[r].copy(), np.searchsorted(col[r], r)
        for q in range(d + 1, n):
            s = s - F[r, q] * v[col[r, q]]
        v[r] = s / F[r, d]
    return v


@pytest.mark.parametrize("N,n,kind", [(5, 2, "around"), (40, 33, "ahead"), (90, 34, "ahead"), (100, 42, "ahead"),
                                      (120, 50, "ahead"), (130, 58, "ahead"), (140, 64, "ahead"), (700, 64, "around"),
                                      (40000, 4, "random"), (20000, 9, "random")])
def test_sweeps_f32(ctx, N, n, kind):
    print(f"case: FP32 sweeps N={N} n={n} {kind}", flush=True)
    rng = np.random.default_rng(N + n)
    st = stencils(rng, N, n, kind)
    w = rng.uniform(-0.5, 0.5, (4, N, n))
    w[0] = rng.uniform(0.0, 0.5, (N, n))
    w[0][:, 0] = -float(n)
    ws, types = [np.ascontiguousarray(w[o]) for o in range(4)], [R.LSFC, R.XSFC, R.YSFC, R.ZSFC]
    e64, e32 = (R.EllOperators(ctx, st, ws, storage=s, types=types) for s in (R.F64, R.F32))
    S = R.Stokes(ctx, e64, e32)
    b = rng.standard_normal(4 * N + 4)
    x = S.gmres(b, tol=1e-30, max_iter=1, krylov=1, mode=R.F32)[0]
    z = b.astype(np.float32)
    z[: 3 * N] = substituted(np.sort(st, axis=1), S.factor().astype(np.float32), z[: 3 * N].reshape(3, N).T).T.reshape(-1)
    z = z.astype(np.float64)
    c = (x @ z) / (z @ z)
    assert c != 0.0
    # two roundings to FP32 of half an ulp (2^-24) each, and the share of them in c
    assert np.max(np.abs(x - c * z) / np.abs(c * z)) < 3.0 * 2.0**-24
    for h in (S, e64, e32):
        h.close()
