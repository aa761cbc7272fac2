"""The windowed CSR product against numpy in FP64, at the edges of its windows (512 entries) and
of its rows per wave (1, 4, 16, 64).

Each row's products are added by up to 64 lanes and then pairwise: the error of a row is at most
(entries) * eps * sum |a_ij x_j|, checked per row with that bound."""
import ctypes as C

import numpy as np
import pytest

import senk_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,lens", [(1, [513]), (3, [0, 1025, 0]), (63, [8]), (64, [8]), (65, [8, 7]), (200, [0, 0, 3]),
                                    (700, [27, 0, 64, 1]), (5000, [7, 600, 1]), (40000, [27]), (140000, [5, 9])])
@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("shift", [0, 1])
def test_rows_and_windows(ctx, N, lens, dt, shift):
    rng = np.random.default_rng(N)
    n = np.resize(np.array(lens), N)
    rptr = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    nnz = int(rptr[-1])
    cind = rng.integers(0, N, nnz).astype(np.int32)
    val, x = rng.uniform(-1, 1, nnz).astype(dt), rng.uniform(-1, 1, N).astype(dt)
    x[0] = 0
    # shift: arrays that start one element into their allocation
    dv, dc = (ctx.array(np.concatenate([np.zeros(shift, t.dtype), t, np.zeros(1, t.dtype)])) for t in (val, cind))
    dr, dx, dy = ctx.array(rptr), ctx.array(x), ctx.array(np.full(N, 9.0, dt))
    S.call("senk_spmv_csr_f64" if dt == np.float64 else "senk_spmv_csr_f32", ctx.h, C.c_void_p(dv.ptr + shift * val.itemsize),
           C.c_void_p(dc.ptr + shift * 4), dr.p, dx.p, dy.p, N)
    prod = val.astype(np.float64) * x.astype(np.float64)[cind]
    rows = np.repeat(np.arange(N), n)
    ref, mag = np.bincount(rows, prod, N), np.bincount(rows, np.abs(prod), N)
    y = dy.download().astype(np.float64)
    assert np.all(np.abs(y - ref) <= (n + 1) * np.finfo(dt).eps * mag)
