"""Stencil search on node sets whose density varies by orders of magnitude: the cells that hold too
many nodes are cut into finer ones. The lists equal the host kd-tree's, and the time stays
near that of an even set."""
import time

import numpy as np
import pytest

import rbffd_gpu_amd as R

pytestmark = pytest.mark.gpu


def sphere(rng, N):
    x = rng.standard_normal((N, 3))
    return x / np.linalg.norm(x, axis=1, keepdims=True)


def graded(rng, N):
    """On the sphere, finer and finer towards the pole."""
    x = sphere(rng, N) * rng.uniform(0.0, 1.0, (N, 1)) ** 4 + np.array([0.0, 0.0, 1.0])
    return x / np.linalg.norm(x, axis=1, keepdims=True)


def cap(rng, N):
    """Half of the nodes on the sphere, half in a cap of 1/50 of its radius."""
    x = sphere(rng, N)
    x[: N // 2] = x[: N // 2] * 0.02 + np.array([0.0, 0.0, 1.0])
    return x / np.linalg.norm(x, axis=1, keepdims=True)


def clusters(rng, N):
    """Volumes of 1, 1e-3 and 1e-5 across, far from each other and inside each other, and one node far away."""
    x = rng.uniform(-1.0, 1.0, (N, 3))
    x[: N // 4] = x[: N // 4] * 1e-3 + np.array([0.3, 0.3, -0.2])
    x[N // 4 : N // 2] = x[N // 4 : N // 2] * 1e-5 + np.array([0.3, 0.3, -0.2])
    x[N // 2 : N // 2 + N // 8] += np.array([3000.0, 0.0, 0.0])
    x[-1] = 1e5
    return x


def deep(rng, N):
    """More halvings than there are levels: a volume of 1e-9 across in one of 1."""
    x = rng.uniform(-1.0, 1.0, (N, 3))
    x[: N // 2] *= 1e-9
    return x


def line(rng, N):
    x = np.zeros((N, 3))
    x[:, 0] = rng.uniform(0.0, 1.0, N) ** 6
    return x


def repeated(rng, N):
    """Every node of a graded set three times, and 300 times the same one."""
    x = np.repeat(graded(rng, N // 3 + 1), 3, axis=0)[:N]
    x[:300] = x[0]
    return x


@pytest.mark.parametrize("k", [1, 17, 50, 169])
@pytest.mark.parametrize("make", [graded, cap, clusters, deep, line, repeated])
def test_graded_sets(ctx, make, k):
    N = 12007 if make is repeated else 30011
    print(f"case: graded search {make.__name__} N={N} k={k}", flush=True)
    rng = np.random.default_rng(N + k)
    xyz = make(rng, N)
    xyz = np.ascontiguousarray(xyz[rng.permutation(N)])
    ref = R.knn_kdtree(xyz, k)
    got, rows = R.knn_gpu(ctx, xyz, k)
    assert np.array_equal(got, ref)
    if make in (graded, cap):
        assert rows < N // 100  # searched here, not left to the host
    d_got, _ = R.knn_gpu_device(ctx, xyz, k)
    assert np.array_equal(d_got.download(), ref)


def test_graded_set_takes_no_other_time_than_an_even_one(ctx):
    """Passes over every node of a few crowded cells took 500 times as long."""
    print("case: time of a graded search", flush=True)
    rng = np.random.default_rng(1)
    N, k = 200000, 31

    def best(xyz):
        xyz = np.ascontiguousarray(xyz[R.order_morton(xyz)])
        t = []
        for _ in range(4):
            t0 = time.perf_counter()
            R.knn_gpu(ctx, xyz, k)
            t.append(time.perf_counter() - t0)
        return min(t)

    even, fine = best(sphere(rng, N)), best(graded(rng, N))
    assert fine < 20 * even, (fine, even)
