"""Many fields per row without a tuned shape: a row's fields have to fit one block, whatever the number of
rows and fields; the largest counts take several fields per thread, and what no block holds is refused."""
import numpy as np
import pytest

import rbffd_gpu_amd as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("F,ops", [(64, 3), (65, 1), (201, 2), (255, 4), (256, 4), (260, 3), (1000, 4), (1024, 1), (2048, 1)])
def test_wide_fields(ctx, F, ops, prec):
    print(f"case: wide F={F} ops={ops} {prec}", flush=True)
    storage = R.F64 if prec == "f64" else R.F32
    dt, eps = (np.float64, 2.0**-53) if prec == "f64" else (np.float32, 2.0**-24)
    N, n = 37, 9
    rng = np.random.default_rng(F + ops)
    idx = rng.integers(0, N, (N, n)).astype(np.int32)
    ws = [rng.standard_normal((N, n)) for _ in range(ops)]
    u = rng.standard_normal((N, F)).astype(dt)
    ell = R.EllOperators(ctx, idx, ws, storage=storage)
    d_u, d_o = ctx.to_device(u), ctx.alloc((ops, N, F), dt)
    ell.spmm(F, d_u, d_o, storage, storage)
    got = d_o.download()
    near = u[idx].astype(np.float64)
    for o, w in enumerate(ws):
        ref = np.einsum("rj,rjf->rf", w, near)
        scale = np.einsum("rj,rjf->rf", np.abs(w), np.abs(near))
        # n products and sums, and FP32 weights moved by up to 1.5 ulp of the row's largest
        bound = (n + 4) * eps * scale + 4 * eps * np.abs(w).max(1)[:, None] * np.abs(near).sum(1)
        assert np.all(np.abs(got[o] - ref) <= bound)
    rk = R.RK4(ctx, ell, F, field_storage=storage, accum=storage)
    rk.set_state(u.astype(np.float64))
    rk.step(1e-3, 5)
    wide = rk.get_state()
    rk.close()
    part = slice(F // 2, F // 2 + 1)  # one field on its own: the same sums in the same order
    rk = R.RK4(ctx, ell, 1, field_storage=storage, accum=storage)
    rk.set_state(np.ascontiguousarray(u[:, part]).astype(np.float64))
    rk.step(1e-3, 5)
    assert np.array_equal(rk.get_state(), wide[:, part])
    rk.close()
    d_u.free()
    d_o.free()
    ell.close()


def test_too_many_fields_refused(ctx):
    idx = np.zeros((8, 1), np.int32)
    ell = R.EllOperators(ctx, idx, [np.ones((8, 1))])
    for F in (257, 514 * 4 + 1, 4096):
        with pytest.raises(R.RbfxError):
            ell.tune_get(1, F, R.F64, R.F64)
    ell.close()
