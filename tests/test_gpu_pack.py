"""The packing kernel's edges: rows per block (chosen from the stencil width), slot chunks above
128, operator groups of four, rows past the end. Applied to unit fields the stored weights come
back exactly, so they are compared bit for bit with the FP64 weights, their nearest FP32 values
and the oracle's row-sum-preserving rounding."""
import numpy as np
import pytest

import oracle as O
import rbffd_gpu_amd as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [R.F64, R.F32, R.F32_RN])
@pytest.mark.parametrize("N,width,n_ops", [(1, 1, 1), (255, 7, 4), (257, 28, 3), (513, 127, 4), (300, 128, 2),
                                           (300, 129, 4), (290, 300, 5), (64, 17, 16)])
def test_packed_weights(ctx, N, width, n_ops, storage):
    print(f"case: pack N={N} n={width} ops={n_ops} storage={storage}", flush=True)
    rng = np.random.default_rng(N * width)
    cols = N + width
    idx = (np.arange(N)[:, None] + np.arange(width)[None, :]).astype(np.int32)
    ws = [rng.standard_normal((N, width)) * 10.0 ** rng.integers(-30, 30, (N, width)) for _ in range(n_ops)]
    ell = R.EllOperators(ctx, idx, ws, n_cols=cols, storage=storage)
    for o in {0, n_ops - 1}:
        if storage == R.F64:
            want = ws[o]
        elif storage == R.F32_RN:
            want = ws[o].astype(np.float32).astype(np.float64)
        else:
            want = O.round_f32_rowsum(ws[o]).astype(np.float64)
        # a unit field at column c picks weight c - row of every row that reaches it
        for c in sorted({0, min(width, cols) - 1, cols - width - 1, cols // 2}):
            u = np.zeros(cols)
            u[c] = 1.0
            d_u, d_o = ctx.to_device(u), ctx.alloc(N, np.float64)
            ell.spmv(o, d_u, d_o, R.F64, R.F64)
            j = c - np.arange(N)
            ok = (j >= 0) & (j < width)
            ref = np.where(ok, want[np.arange(N), np.clip(j, 0, width - 1)], 0.0)
            assert np.array_equal(d_o.download(), ref)
            d_u.free()
            d_o.free()
    ell.close()
