"""Device memory that a context keeps for its next objects is given back on request, and when another
context on the device runs out of it."""
import ctypes as C

import numpy as np
import pytest

import rbffd_gpu_amd as R

pytestmark = pytest.mark.gpu
MiB = 1 << 20


def mem_info():
    free, total = C.c_size_t(), C.c_size_t()
    assert R.load_library().hipMemGetInfo(C.byref(free), C.byref(total)) == 0  # the HIP runtime the library uses
    return free.value, total.value


def build(ctx, N, n):
    """An operator set of at least N * n * 12 bytes, applied once and dropped."""
    idx = ((np.arange(N)[:, None] + np.arange(n)[None, :]) % N).astype(np.int32)
    w = np.random.default_rng(N).standard_normal((N, n))
    d_idx, d_w = ctx.to_device(idx), ctx.to_device(w)
    ell = R.EllOperators(ctx, d_idx, [d_w])
    d_u, d_o = ctx.to_device(np.cos(np.arange(N))), ctx.alloc((N,), np.float64)
    ell.spmv(0, d_u, d_o)
    out = d_o.download()
    ell.close()
    for d in (d_idx, d_w, d_u, d_o):
        d.free()
    return out


def test_release_idle():
    print("case: release idle memory", flush=True)
    N, n = 400000, 31
    with R.Context(0) as c:
        first = build(c, N, n)
        before, _ = mem_info()
        given = c.release_idle()
        assert given >= N * n * 12
        assert mem_info()[0] - before >= N * n * 12 - 4 * MiB
        assert c.release_idle() == 0
        assert np.array_equal(build(c, N, n), first)  # the context works on


def test_idle_memory_serves_another_context_that_runs_out():
    print("case: idle memory of another context", flush=True)
    N, n = 400000, 31
    with R.Context(0) as a, R.Context(0) as b:
        first = build(a, N, n)
        before, total = mem_info()
        p = C.c_void_p()
        assert R.RBFX.rbfx_dev_alloc(b.h, 2 * total, C.byref(p)) == -3 and not p.value  # RBFX_E_NOMEM
        assert mem_info()[0] - before >= N * n * 12 - 4 * MiB
        assert a.release_idle() == 0
        assert np.array_equal(build(a, N, n), first)
