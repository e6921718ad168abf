"""Weight solves at the edges of the matrix-core layouts, and with few and many right-hand sides."""
import numpy as np
import pytest

import rbffd_gpu_amd as R

pytestmark = pytest.mark.gpu

T_MASKS = {1: R.X, 4: R.X | R.Y | R.Z | R.LAPL, 5: R.X | R.Y | R.Z | R.LAPL | R.HV,
           9: R.X | R.Y | R.Z | R.LAPL | R.HV | R.R | R.XSFC | R.YSFC | R.ZSFC}


@pytest.fixture(scope="module")
def ctx():
    with R.Context(0) as c:
        yield c


@pytest.mark.parametrize("T", sorted(T_MASKS))
def test_weights_at_layout_edges(ctx, monkeypatch, T):
    """Systems of 16 j and 16 j +- 1 unknowns, the smallest and the largest: the matrix-core solver and
    the register-resident one do the same operations per element, so weights and diagnostics are equal
    bit for bit; a call without diagnostics gives the same weights."""
    m_list = [2, 3, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 95, 96, 97, 111, 112, 113, 120]
    print("case: layout edges, T", T, flush=True)
    N = 5000
    xyz = R.nodes_fibonacci(N, 1e-3, 2)
    rng = np.random.default_rng(T)
    nn = np.repeat([m - 1 for m in m_list], 3)  # degree 0: one polynomial row
    rng.shuffle(nn)
    rows = rng.choice(N, size=nn.size, replace=False)
    knn = R.knn_kdtree(xyz, 119)
    off = np.concatenate([[0], np.cumsum(nn)]).astype(np.int32)
    idx = np.concatenate([knn[r, :k] for r, k in zip(rows, nn)]).astype(np.int32)
    eps = np.full(nn.size, 5.0)
    kw = dict(dim=3, poly_deg=0, hv_k=2, hv_scale=-1e-3)
    monkeypatch.delenv("RBFX_WEIGHTS_F64", raising=False)
    w, dg = ctx.weights(off, idx, xyz, eps, T_MASKS[T], diag=True, **kw)
    w0, _ = ctx.weights(off, idx, xyz, eps, T_MASKS[T], **kw)
    monkeypatch.setenv("RBFX_WEIGHTS_F64", "reg")
    w_ref, dg_ref = ctx.weights(off, idx, xyz, eps, T_MASKS[T], diag=True, **kw)
    assert w.shape[0] == T and np.isfinite(w).all()
    assert np.array_equal(w, w_ref) and np.array_equal(dg, dg_ref)
    assert np.array_equal(w, w0)
