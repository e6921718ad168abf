"""The GPU stencil search at the edges of its grid and its candidate lists: few nodes, all nodes in
one cell, lines (many cells along one axis), clusters of very different density (searches that
grow, and bounds that are narrowed), far outliers, extents that over- and underflow, repeated
nodes by the hundred, the longest lists. Lists equal the host kd-tree's, and the rows handed back
are those with equal distances among their k+1 nearest."""
import numpy as np
import pytest

import rbffd_gpu_amd as R

pytestmark = pytest.mark.gpu


def nodes(name):
    rng = np.random.default_rng(len(name))
    x = rng.random((1500, 3))
    if name == "two":
        return x[:2]
    if name == "line":
        return np.outer(rng.random(2000), [1.0, 0.0, 0.0])
    if name == "diagonal":
        return np.outer(rng.random(2000), [1.0, 2.0, 3.0])
    if name == "clusters":
        return np.concatenate([x[:700] * 1e-6, x[700:1400] * 1e-2 + 5.0, x[1400:] * 100.0])
    if name == "outlier":
        return np.concatenate([x, [[1e5, -1e5, 1e5]]])
    if name == "huge":
        return x * 1e200
    if name == "tiny":
        return x * 1e-200
    if name == "repeated":
        return np.concatenate([x[:300], np.repeat(x[300:303], 400, axis=0)])
    if name == "lattice":
        return np.stack(np.meshgrid(*[np.arange(12.0)] * 3), -1).reshape(-1, 3)
    return x


def ties(xyz, k):
    """Rows with equal distances among their k+1 nearest."""
    with np.errstate(over="ignore", under="ignore"):
        d = np.zeros((len(xyz), len(xyz)))
        for c in range(3):
            d = d + (xyz[:, None, c] - xyz[None, :, c]) ** 2
    d = np.sort(np.partition(d, k, axis=1)[:, : k + 1], axis=1)
    return int((d[:, 1:] == d[:, :-1]).any(1).sum())


@pytest.mark.parametrize("name,k", [("two", 1), ("cube", 1), ("cube", 63), ("cube", 64), ("cube", 127), ("cube", 169),
                                    ("cube", 170), ("line", 31), ("diagonal", 50), ("clusters", 50), ("outlier", 17),
                                    ("huge", 9), ("tiny", 9), ("repeated", 30), ("lattice", 27)])
def test_knn_edges(ctx, name, k):
    print(f"case: knn {name} k={k}", flush=True)
    xyz = np.ascontiguousarray(nodes(name))
    got, n_host = R.knn_gpu(ctx, xyz, k)
    assert np.array_equal(got, R.knn_kdtree(xyz, k))
    assert n_host == (len(xyz) if k >= 170 else ties(xyz, k))
    d_st, n_dev = R.knn_gpu_device(ctx, xyz, k)
    assert n_dev == n_host and np.array_equal(d_st.download(), got)
    d_st.free()


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("at", [0, 3 * 999 + 2])
def test_knn_non_finite(ctx, bad, at):
    xyz = np.random.default_rng(0).random((1000, 3))
    xyz.reshape(-1)[at] = bad
    with pytest.raises(R.RbfxError, match="non-finite"):
        R.knn_gpu(ctx, xyz, 9)
