"""The ILU(0) sweeps at the edges of their kernel: every variant of entries per side (32, 40, 48,
56 and 64), levels of more rows than a chunk, chunks of one row, fewer chunks than waves, and values
older than the ring in LDS (more than 16384 tasks back). Factor and sweeps equal the CPU
restatement bit for bit."""
import numpy as np
import pytest

import oracle as O
import rbffd_gpu_amd as R

pytestmark = pytest.mark.gpu


def stencils(rng, N, n, kind):
    if kind == "random":  # few levels, long reaches
        st = rng.integers(0, N - 1, (N, n))
        for i in range(N):
            while len(set(st[i, 1:].tolist())) < n - 1:
                st[i] = rng.integers(0, N - 1, n)
        st += st >= np.arange(N)[:, None]  # any node but the centre
    else:  # the rows before and after, wrapped
        st = (np.arange(N)[:, None] + np.arange(n)[None, :] - (n // 2 if kind == "around" else 0)) % N
        st[:, [0, n // 2 if kind == "around" else 0]] = st[:, [n // 2 if kind == "around" else 0, 0]]
    st[:, 0] = np.arange(N)
    return np.ascontiguousarray(st.astype(np.int32))


@pytest.mark.parametrize("N,n,kind", [(5, 2, "around"), (40, 33, "ahead"), (90, 34, "ahead"), (100, 41, "ahead"),
                                      (100, 42, "ahead"), (120, 49, "ahead"), (120, 50, "ahead"), (130, 57, "ahead"),
                                      (130, 58, "ahead"), (140, 64, "ahead"), (700, 64, "around"), (40000, 4, "random"),
                                      (20000, 9, "random")])
def test_sweep_edges(ctx, N, n, kind):
    print(f"case: sweeps N={N} n={n} {kind}", flush=True)
    rng = np.random.default_rng(N + n)
    st = stencils(rng, N, n, kind)
    w = rng.uniform(-0.5, 0.5, (4, N, n))
    w[0] = rng.uniform(0.0, 0.5, (N, n))
    w[0][:, 0] = -float(n)
    e64 = R.EllOperators(ctx, st, [np.ascontiguousarray(w[o]) for o in range(4)], storage=R.F64,
                         types=[R.LSFC, R.XSFC, R.YSFC, R.ZSFC])
    S = R.Stokes(ctx, e64)
    A = O.stokes_assemble(st, w)
    F = O.ilu0(A, 0, 3 * N)
    assert np.array_equal(S.factor(), F.data[: F.indptr[N]].reshape(N, n))
    for scale in (1.0, 1e-300):
        v = rng.standard_normal(A.n) * scale
        assert np.array_equal(S.precond(v), O.ilu0_apply(F, v))
    S.close()
    e64.close()
