"""GMRES(m)'s two-pass modified Gram-Schmidt against the oracle's column-by-column one.

The coefficients are the same in exact arithmetic; in FP64 they differ by a few roundings per
inner product, so the residual estimates of the first cycles agree to far better than 1e-8
relative while they are large against the rounding level (here above 1e-8 of the first).
"""
import ctypes as C

import numpy as np
import pytest

import senk_amd as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# accumulator counts of the dots pass (8, 16, 24, 32), two chunks (33, 50, 64), and the launch
# per column (65)
@pytest.mark.parametrize("m", [1, 8, 9, 17, 25, 32, 33, 50, 64, 65])
def test_residual_history_matches_the_oracle(ctx, m):
    rptr, cind, val = S.gen_convdiff27(11, 10.0)
    N = len(rptr) - 1
    x = S.gen_uniform(3, N)
    b = np.zeros(N)
    O.orc().or_spmv_csr_d(O.P(val), O.P(cind), O.P(rptr), O.P(x), O.P(b), N)
    nrm_b, cap = float(np.linalg.norm(b)), 70
    outer, eps = -(-cap // m), 1e-30  # run the whole budget, unpreconditioned (slow convergence)
    ho, hd = np.zeros(outer * m), np.zeros(outer * m)
    xo, conv = np.zeros(N), C.c_int()
    spec = O.prec_spec(0)
    O.orc().or_gmres_d(O.P(val), O.P(cind), O.P(rptr), C.byref(spec), O.P(b), O.P(xo), nrm_b, outer, m, N, eps,
                       O.P(ho), len(ho), C.byref(conv))
    dv, dc, dr, db, dx = ctx.array(val), ctx.array(cind), ctx.array(rptr), ctx.array(b), ctx.zeros(N)
    res = S.senk_result()
    S.call("senk_gmresm_f64", ctx.h, dv.p, dc.p, dr.p, db.p, dx.p, C.c_double(nrm_b), outer, m, N, C.c_double(eps), 0,
           C.byref(res), O.P(hd), len(hd))
    big = ho > 1e-8 * ho[0]
    assert big.sum() >= min(30, len(ho))
    assert np.max(np.abs(hd[big] - ho[big]) / ho[big]) <= 1e-8


# one lane per row of the cycle end's triangular solve up to 64 columns, several beyond
@pytest.mark.parametrize("m", [1, 2, 63, 64, 65, 128, 129])
def test_solution_of_one_cycle_matches_the_oracle(ctx, m):
    # x = V y is the minimiser over the Krylov space: its error is a few roundings times the
    # condition number (below 1e3 here), far below 1e-9 relative
    rptr, cind, val = S.gen_convdiff27(20, 10.0)
    N = len(rptr) - 1
    x = S.gen_uniform(5, N)
    b = np.zeros(N)
    O.orc().or_spmv_csr_d(O.P(val), O.P(cind), O.P(rptr), O.P(x), O.P(b), N)
    nrm_b, eps = float(np.linalg.norm(b)), 1e-30
    ho, hd = np.zeros(m), np.zeros(m)
    xo, conv = np.zeros(N), C.c_int()
    spec = O.prec_spec(0)
    O.orc().or_gmres_d(O.P(val), O.P(cind), O.P(rptr), C.byref(spec), O.P(b), O.P(xo), nrm_b, 1, m, N, eps,
                       O.P(ho), len(ho), C.byref(conv))
    dv, dc, dr, db, dx = ctx.array(val), ctx.array(cind), ctx.array(rptr), ctx.array(b), ctx.zeros(N)
    res = S.senk_result()
    S.call("senk_gmresm_f64", ctx.h, dv.p, dc.p, dr.p, db.p, dx.p, C.c_double(nrm_b), 1, m, N, C.c_double(eps), 0,
           C.byref(res), O.P(hd), len(hd))
    assert np.linalg.norm(dx.download() - xo) <= 1e-9 * np.linalg.norm(xo)


# the dots pass reduces two sets of products one after the other through one LDS buffer; all
# reductions run in a fixed order, so repeated solves give the same bits
@pytest.mark.parametrize("m", [8, 30, 50])
def test_repeated_solves_give_the_same_bits(ctx, m):
    rptr, cind, val = S.gen_convdiff27(33, 10.0)
    N = len(rptr) - 1
    b = S.gen_uniform(7, N)
    nrm_b = float(np.linalg.norm(b))
    d = [ctx.array(t) for t in (val, cind, rptr, b)]
    first = None
    for _ in range(30):
        dx, hd, res = ctx.zeros(N), np.zeros(m), S.senk_result()
        S.call("senk_gmresm_f64", ctx.h, *(t.p for t in d), dx.p, C.c_double(nrm_b), 1, m, N, C.c_double(1e-30), 0,
               C.byref(res), O.P(hd), len(hd))
        got = (hd, dx.download())
        first = first or got
        assert np.array_equal(got[0], first[0]) and np.array_equal(got[1], first[1])
