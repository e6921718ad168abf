"""One field on four lanes per row (share 6): same bits as a lane per row, for SpMM / SpMV and RK4,
at the edges of its 16-row waves and 32-slot chunks, for every operator count and precision, with
and without a row order and coefficients; and the default shape of small sets reports it."""
import numpy as np
import pytest

import rbffd_gpu_amd as R
from rbffd_gpu_amd import tune as TU

pytestmark = pytest.mark.gpu

PRECISIONS = {"f64": (R.F64, R.F64, R.F64), "f32": (R.F32, R.F32, R.F32), "f32_sum64": (R.F32, R.F32, R.F64),
              "f32_f64": (R.F32, R.F64, R.F64)}


@pytest.mark.parametrize("prec", list(PRECISIONS))
@pytest.mark.parametrize("N,n,ops", [(1, 1, 1), (15, 3, 2), (16, 4, 3), (17, 5, 4), (257, 31, 4), (300, 32, 3),
                                     (301, 33, 2), (500, 64, 1), (333, 101, 3)])
def test_quad_bit_identical(ctx, N, n, ops, prec):
    print(f"case: quad N={N} n={n} ops={ops} {prec}", flush=True)
    storage, ft, acc = PRECISIONS[prec]
    rng = np.random.default_rng(N + n)
    idx = rng.integers(0, N, (N, n)).astype(np.int32)
    ws = [rng.standard_normal((N, n)) for _ in range(ops)]
    u = rng.standard_normal((N, 1))
    for order in (None, rng.permutation(N)):
        ell = R.EllOperators(ctx, idx, ws, storage=storage)
        if order is not None:
            ell.set_row_order(order.astype(np.int32))
        d_u = ctx.to_device(u.astype(np.float64 if ft == R.F64 else np.float32))
        out, state = [], []
        for share in (0, 6):
            ell.tune_set(TU.KIND_SPMM, 1, ft, acc, 1, 64, 8, share)
            d_o = ctx.alloc((ops, N, 1), d_u.dtype)
            ell.spmm(1, d_u, d_o, ft, acc)
            out.append(d_o.download())
            d_o.free()
            if prec == "f32_f64":
                continue  # FP32 operators step FP32 stage fields only
            ell.tune_set(TU.KIND_RK4, 1, ft, acc, 1, 64, 8, share)
            coefs = [None if o == 1 else np.cos(np.arange(N) + o) for o in range(ops)]
            rk = R.RK4(ctx, ell, 1, field_storage=ft, accum=acc, coefs=coefs)
            rk.set_state(u)
            rk.step(1e-3, 3)
            state.append(rk.get_state())
            rk.close()
        assert np.array_equal(out[0], out[1])
        assert prec == "f32_f64" or np.array_equal(state[0], state[1])
        R.RBFX.rbfx_tune_clear()
        d_u.free()
        ell.close()


def test_quad_is_the_small_default(ctx):
    idx = np.tile(np.arange(31, dtype=np.int32), (64, 1))
    ell = R.EllOperators(ctx, idx, [np.ones((64, 31))] * 3)
    assert ell.tune_get(TU.KIND_RK4, 1, R.F64, R.F64) == (1, 64, 8, 6)
    ell.tune_set(TU.KIND_RK4, 1, R.F64, R.F64, *ell.tune_get(TU.KIND_RK4, 1, R.F64, R.F64))  # taken back as given
    for args in ((2, 1, 64, 8), (1, 1, 128, 8), (1, 1, 64, 4)):
        with pytest.raises(R.RbfxError):
            ell.tune_set(TU.KIND_RK4, args[0], R.F64, R.F64, *args[1:], 6)
    ell.close()
