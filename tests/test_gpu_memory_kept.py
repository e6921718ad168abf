"""What a context keeps of dropped objects' memory: at most 32 blocks and 1/64 of the device's memory; and Stokes
solvers, weights and searches on blocks that held NaN weights give the results of a fresh context."""
import numpy as np
import pytest

import rbffd_gpu_amd as R
from test_gpu_idle_memory import mem_info

pytestmark = pytest.mark.gpu


def drop_set(ctx, N, n, ops, value):
    """Builds and drops a set of N * n * (4 + 8 * ops) bytes whose weights are all `value`."""
    d_idx, d_w = ctx.to_device(np.zeros((N, n), np.int32)), ctx.to_device(np.full((N, n), value))
    R.EllOperators(ctx, d_idx, [d_w] * ops).close()
    d_idx.free()
    d_w.free()


def test_blocks_are_bounded():
    print("case: kept blocks", flush=True)
    # two blocks each, of 68 and 136 bytes a row: less than twice as many rows in the last set as in the
    # first, so that no block is as large as a later one asks for
    rows = [98304 + 2048 * i for i in range(40)]
    with R.Context(0) as c:
        for N in rows:
            drop_set(c, N, 17, 1, 0.0)
        assert c.release_idle() == sum(rows[-16:]) * 17 * 12


def test_bytes_are_bounded():
    print("case: kept bytes", flush=True)
    with R.Context(0) as c:
        for i in range(5):  # 1.2 to 3.4 GB
            drop_set(c, int(300000 * 1.3**i), 31, 16, 0.0)
        assert mem_info()[1] // 160 < c.release_idle() <= mem_info()[1] // 64


def results(ctx):
    """Factor, preconditioned vector and GMRES solutions of a Stokes system, weights, stencils."""
    N, n = 4800, 31
    xyz = R.nodes_fibonacci(N, 1e-3, 0)
    xyz = np.ascontiguousarray(xyz[R.order_morton(xyz)])
    st, _ = R.knn_gpu(ctx, xyz, n)
    off, idx = R.csr_from_fixed(st)
    w, _ = ctx.weights(off, idx, xyz, 0.035 * np.sqrt(N) - 0.1, R.LSFC | R.XSFC | R.YSFC | R.ZSFC)
    many = R.nodes_fibonacci(150000, 1e-4, 1)  # enough stencils for a scratch of more than 1 MiB
    far, _ = R.knn_gpu(ctx, many, 17)
    w_far, _ = ctx.weights(*R.csr_from_fixed(far), many, 0.026 * np.sqrt(150000.0) - 0.08, R.X)
    ws, types = [np.ascontiguousarray(v.reshape(N, n)) for v in w], [R.LSFC, R.XSFC, R.YSFC, R.ZSFC]
    e64, e32 = (R.EllOperators(ctx, st, ws, storage=s, types=types) for s in (R.F64, R.F32))
    S = R.Stokes(ctx, e64, e32)
    b = np.concatenate([np.cos(3.0 * xyz.T.reshape(-1)), np.zeros(N + 4)])
    out = [st, w, far, w_far, S.factor(), S.precond(b), S.apply(b)]
    for mode in (R.F64, R.F32):
        out.append(S.gmres(b, tol=1e-10, max_iter=12, krylov=12, mode=mode)[0])
    for h in (S, e64, e32):
        h.close()
    return out


def test_results_on_blocks_that_held_nan():
    print("case: blocks that held NaN", flush=True)
    with R.Context(0) as c:
        fresh = results(c)
    with R.Context(0) as c:
        for _ in range(2):
            for i in range(24):  # 1 MiB and up to 170 MiB: a block for whatever is asked for next
                drop_set(c, int(1.25**i * (1 << 20) / (16 * 16 * 8)) + 1, 16, 16, np.nan)
            for got, ref in zip(results(c), fresh):
                assert np.array_equal(got, ref)
    assert all(np.isfinite(v).all() for v in fresh)
