"""Device memory that operator sets, their tables, the Stokes factor and the searches hand on to each other:
results do not depend on what a block held before, and what is kept is bounded and given back."""
import ctypes as C

import numpy as np
import pytest

import rbffd_gpu_amd as R

pytestmark = pytest.mark.gpu


def _apply(ctx, N, n, ops, seed, storage, order):
    rng = np.random.default_rng(seed)
    idx = ((np.arange(N)[:, None] + rng.integers(0, 40, (N, n))) % N).astype(np.int32)
    ws = [rng.standard_normal((N, n)) for _ in range(ops)]
    u = rng.standard_normal((N, 16)).astype(np.float64 if storage == R.F64 else np.float32)
    ell = R.EllOperators(ctx, idx, ws, storage=storage)
    if order:
        ell.set_row_order(rng.permutation(N).astype(np.int32))
    ell.build_local(64, 1024)
    d_u, d_o = ctx.to_device(u), ctx.alloc((ops, N, 16), u.dtype)
    ell.spmm(16, d_u, d_o, storage, storage)
    out = d_o.download()
    ell.close()
    d_u.free()
    d_o.free()
    return out


# sizes around the smallest block kept (1 MiB), shrinking and growing, so that blocks are taken over by
# sets that fill them partly
CASES = [(20011, 31, 4, R.F64, False), (18000, 31, 4, R.F64, True), (8192, 32, 3, R.F32, False), (8193, 32, 3, R.F32, False),
         (20000, 31, 4, R.F32, True), (17001, 37, 3, R.F64, False), (20011, 31, 4, R.F64, True)]


def test_results_do_not_depend_on_earlier_blocks(ctx):
    fresh = []
    for i, (N, n, ops, st, order) in enumerate(CASES):
        with R.Context(0) as c:
            fresh.append(_apply(c, N, n, ops, i, st, order))
    for _ in range(2):
        for i, (N, n, ops, st, order) in enumerate(CASES):
            print(f"case: reuse {i}", flush=True)
            assert np.array_equal(_apply(ctx, N, n, ops, i, st, order), fresh[i])


def test_kept_memory_is_bounded_and_given_back():
    def mem_info():
        free, total = C.c_size_t(), C.c_size_t()
        assert R.load_library().hipMemGetInfo(C.byref(free), C.byref(total)) == 0  # the HIP runtime the library uses
        return free.value, total.value

    def work(c, sizes):
        for N in sizes:
            idx = np.zeros((N, 17), np.int32)
            R.EllOperators(c, idx, [np.zeros((N, 17))]).close()
        xyz = np.random.default_rng(0).standard_normal((200000, 3))
        lists = [R.knn_gpu(c, xyz, 17)[0] for _ in range(3)]
        assert all(np.array_equal(lists[0], v) for v in lists[1:])

    with R.Context(0) as c:
        work(c, [9000])  # the runtime's own allocations
    free0, total = mem_info()
    with R.Context(0) as c:
        work(c, [9000 + 4000 * i for i in range(40)])  # more sizes than blocks are kept, none serving the next
        free1, _ = mem_info()
        assert free0 - free1 <= total // 64 + (256 << 20)
    free2, _ = mem_info()
    assert free0 - free2 <= 256 << 20
