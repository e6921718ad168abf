"""Tile tables of the LDS-staged gathers (rbfx_ell_build_local) at the sizes where the device
build can go wrong: short and long last tiles, chunk edges, caps that cut after one row, the
widest stencils its LDS tables take and the first that go to the host, lists of scattered
nodes. The tiles are those of the greedy cut restated here, and the staged SpMM through the
tables equals the direct gathers bit for bit."""
import numpy as np
import pytest

import rbffd_gpu_amd as R
from rbffd_gpu_amd import tune as TU

pytestmark = pytest.mark.gpu


def greedy(idx, lt, cap):
    """(longest list, tiles) of the cut: chunks of 64 lt rows, tiles of at most lt rows and cap nodes."""
    k_max = tiles = 0
    for lo in range(0, len(idx), 64 * lt):
        hi = min(len(idx), lo + 64 * lt)
        p = lo
        while p < hi:
            u, start = set(), p
            while p < hi and p - start < lt:
                m = u | set(idx[p].tolist())
                if cap > 0 and p > start and len(m) > cap:
                    break
                u, p = m, p + 1
            k_max, tiles = max(k_max, len(u)), tiles + 1
    return k_max, tiles


@pytest.mark.parametrize("N,width,lt,cap,scattered", [
    (1, 1, 32, 0, False), (31, 1, 32, 1, False), (300, 7, 32, 7, False), (2048, 5, 32, 20, False),
    (2049, 5, 32, 0, False), (8193, 50, 128, 768, False), (4097, 33, 64, 90, False), (700, 112, 128, 0, False),
    (700, 113, 128, 200, False), (900, 448, 32, 0, False), (900, 449, 32, 0, False), (5000, 31, 128, 0, True),
    (5000, 31, 64, 31, True), (20000, 64, 128, 0, True), (40000, 100, 128, 0, True)])
def test_local_tables(ctx, N, width, lt, cap, scattered):
    print(f"case: local tables N={N} n={width} tile={lt} cap={cap} scattered={scattered}", flush=True)
    rng = np.random.default_rng(N + width)
    width = min(width, N)
    if scattered:
        idx = rng.integers(0, N, (N, width))
    else:  # a window around the row, in another order per row
        idx = (np.arange(N)[:, None] + rng.permuted(np.tile(np.arange(width), (N, 1)), axis=1)) % N
    idx[:, 0] = np.arange(N)
    idx = idx.astype(np.int32)
    ws = [rng.standard_normal((N, width)) for _ in range(3)]
    ell = R.EllOperators(ctx, idx, ws, storage=R.F64)
    tl, k_max, n_tiles = ell.build_local(lt, cap)
    assert (tl, k_max, n_tiles) == (lt, *greedy(idx, lt, cap))
    if k_max * 16 * 8 <= TU.LDS_BYTES:
        d_u = ctx.to_device(rng.standard_normal((N, 16)))
        outs = []
        for block, share in ((256, 0), (lt * 4, 4)):
            ell.tune_set(TU.KIND_SPMM, 16, R.F64, R.F64, 4, block, 4, share)
            d_o = ctx.alloc((3, N, 16), np.float64)
            ell.spmm(16, d_u, d_o)
            outs.append(d_o.download())
            d_o.free()
        assert np.array_equal(outs[0], outs[1])
        d_u.free()
    ell.close()
