"""Single-launch triangular solves on the caller's CSR and BCSR factors (ABMC colors and
plans).

Every row keeps the sequential solve's operations and their order, so the results must be the
oracle's sequential solve bit for bit, whatever solves of other sizes and types ran before
on the context (the solves share two vectors that each leaves ready for the next).
"""
import ctypes as C

import numpy as np
import pytest

import senk_amd as S
from oracle import oracle as O
from tests.helpers import abmc_system, ilu_factors, oracle_ilu0, relerr

pytestmark = pytest.mark.gpu


def _seq(L, U, x):
    """The oracle's sequential solves L, then U, in x's type."""
    N, s = len(x), "d" if x.dtype == np.float64 else "f"
    yl, yu = np.zeros_like(x), np.zeros_like(x)
    getattr(O.orc(), "or_sptrsv_l_" + s)(O.P(L[0]), O.P(L[1]), O.P(L[2]), O.P(x), O.P(yl), N)
    getattr(O.orc(), "or_sptrsv_u_" + s)(O.P(U[0]), O.P(U[1]), O.P(U[2]), O.P(yl), O.P(yu), N)
    return yl, yu


def _typed(f, dt):
    return (np.ascontiguousarray(f[0].astype(dt)), f[1], f[2])


def _abmc_case(ctx, mat, bsize, method, dt):
    val, cind, rptr, N = S.padding(mat[2], mat[1], mat[0], bsize, len(mat[0]) - 1)
    sy = abmc_system(rptr, cind, val, bsize, method)
    L, U = (_typed(f, dt) for f in ilu_factors(sy))
    x = np.random.default_rng(N + bsize).uniform(-1, 1, N).astype(dt)
    x[N // 3] = 0.0
    yl, yu = _seq(L, U, x)
    d = [ctx.array(t) for t in (*L, *U, x)]
    s = "f64" if dt == np.float64 else "f32"
    cp = O.P(sy["cptr"])
    dy = ctx.zeros(N, dt)
    S.call("senk_sptrsv_csr_l_abmc_" + s, ctx.h, *(t.p for t in d[:3]), d[6].p, dy.p, N, cp, sy["nc"], bsize)
    t = dy.download()
    S.call("senk_sptrsv_csr_u_abmc_" + s, ctx.h, *(t.p for t in d[3:6]), dy.p, dy.p, N, cp, sy["nc"], bsize)  # in place
    assert np.array_equal(t, yl) and np.array_equal(dy.download(), yu)


def _plan_case(ctx, mat, dt):
    rptr, cind, val = mat
    N = len(rptr) - 1
    L, U = (_typed(f, dt) for f in ilu_factors(dict(val=val, cind=cind, rptr=rptr)))
    x = np.random.default_rng(N).uniform(-1, 1, N).astype(dt)
    yl, yu = _seq(L, U, x)
    d = [ctx.array(t) for t in (*L, *U, x)]
    s = "f64" if dt == np.float64 else "f32"
    plans = []
    for f, up in ((L, 0), (U, 1)):
        p = C.c_void_p()
        S.call("senk_trsv_plan_create", ctx.h, O.P(f[2]), O.P(f[1]), N, up, C.byref(p))
        plans.append(p)
    dy = d[6]  # L in place as well
    S.call("senk_sptrsv_csr_l_" + s, ctx.h, plans[0], *(t.p for t in d[:3]), dy.p, dy.p, N)
    t = dy.download()
    S.call("senk_sptrsv_csr_u_" + s, ctx.h, plans[1], *(t.p for t in d[3:6]), dy.p, dy.p, N)
    u = dy.download()
    for p in plans:
        S.lib().senk_trsv_plan_destroy(p)
    assert np.array_equal(t, yl) and np.array_equal(u, yu)


def _tridiagonal(n):
    r = np.arange(n)
    rows = np.concatenate([r, r[1:], r[:-1]])
    cols = np.concatenate([r, r[1:] - 1, r[:-1] + 1])
    vals = np.concatenate([np.full(n, 4.0), np.full(n - 1, -1.0), np.full(n - 1, -1.5)])
    o = np.lexsort((cols, rows))
    rptr = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))])
    return rptr.astype(np.int32), cols[o].astype(np.int32), vals[o]


def _chain_then_wide(chain, wide):
    """`chain` levels of one row, then one of `wide` rows that wait for the last of them: on all
    XCDs, most of whose streams have nothing in the chain's levels."""
    rows = [[i - 1, i] if 0 < i < chain else [i] if i == 0 else [chain - 1, i] for i in range(chain + wide)]
    rptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    cind = np.concatenate(rows).astype(np.int32)
    val = np.where(cind == np.repeat(np.arange(len(rows)), np.diff(rptr)), 3.0, -1.0)
    return rptr, cind, val


# sizes around the slice of 64 rows and the ticket of 4 slices, rows of more than one round of
# gathers, slices of more entries than the wave stages in LDS (27-point in FP64)
@pytest.mark.parametrize("bsize", [1, 2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_abmc_in_turn_with_other_sizes(ctx, bsize, dt):
    other = np.float32 if dt == np.float64 else np.float64
    _abmc_case(ctx, S.gen_convdiff27(11, 10.0), bsize, "connect", dt)
    _abmc_case(ctx, S.gen_poisson7(3, 5, 4), bsize, "simple", other)
    _abmc_case(ctx, S.gen_vardiff7(13, 3, 4.0, 1.5), bsize, "simple", dt)
    _abmc_case(ctx, S.gen_unstructured(2500, 5), bsize, "connect", dt)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_plans_in_turn_with_other_sizes(ctx, dt):
    other = np.float32 if dt == np.float64 else np.float64
    _plan_case(ctx, S.gen_poisson7(13, 9, 11), dt)        # one stream
    _plan_case(ctx, _tridiagonal(1), other)
    empty = C.c_void_p()
    S.call("senk_trsv_plan_create", ctx.h, O.P(np.zeros(1, np.int32)), O.P(np.zeros(1, np.int32)), 0, 0, C.byref(empty))
    S.call("senk_sptrsv_csr_l_f64", ctx.h, empty, None, None, None, None, None, 0)
    S.lib().senk_trsv_plan_destroy(empty)
    _plan_case(ctx, _tridiagonal(333), dt)                # every row waits on one of its own wave
    _plan_case(ctx, S.gen_convdiff27(12, 10.0), dt)       # rows of 13
    _plan_case(ctx, S.gen_unstructured(20000, 7), dt)     # long rows, several rounds
    _plan_case(ctx, S.gen_poisson7(48, 46, 47), other)    # eight streams


def test_non_finite_values_pass_through(ctx):
    """An x that holds NaN (with any payload, the sentinel's too) and infinities: the solve
    ends, and what it leaves non-finite is what the sequential solve leaves."""
    rptr, cind, val = S.gen_poisson7(12)
    N = len(rptr) - 1
    sy = abmc_system(rptr, cind, val, 8)
    L, U = ilu_factors(sy)
    x = np.random.default_rng(4).uniform(-1, 1, N)
    x[5], x[700] = np.inf, np.nan
    x.view(np.uint64)[901] = 0x7FF4A5A5A5A5A5A5
    yl, yu = _seq(L, U, x)
    d = [ctx.array(t) for t in (*L, *U, x)]
    dy = ctx.zeros(N)
    cp = O.P(sy["cptr"])
    S.call("senk_sptrsv_csr_l_abmc_f64", ctx.h, *(t.p for t in d[:3]), d[6].p, dy.p, N, cp, sy["nc"], 8)
    assert np.array_equal(dy.download(), yl, equal_nan=True)
    S.call("senk_sptrsv_csr_u_abmc_f64", ctx.h, *(t.p for t in d[3:6]), dy.p, dy.p, N, cp, sy["nc"], 8)
    assert np.array_equal(dy.download(), yu, equal_nan=True)
    _abmc_case(ctx, (rptr, cind, val), 8, "connect", np.float64)  # nothing is left behind


def test_schedules_outside_the_single_launch(ctx):
    """More levels than the launch's table holds, and colors that stop short of N, keep the
    launch per level."""
    rptr, cind, val = _tridiagonal(400)
    N = len(rptr) - 1
    L, U = ilu_factors(dict(val=val, cind=cind, rptr=rptr))
    x = np.random.default_rng(2).uniform(-1, 1, N)
    yl, yu = _seq(L, U, x)
    d = [ctx.array(t) for t in (*L, *U, x)]
    dy = ctx.zeros(N)
    cptr = np.arange(N + 1, dtype=np.int32)  # one row a color
    S.call("senk_sptrsv_csr_l_amc_f64", ctx.h, *(t.p for t in d[:3]), d[6].p, dy.p, N, O.P(cptr), N)
    S.call("senk_sptrsv_csr_u_amc_f64", ctx.h, *(t.p for t in d[3:6]), dy.p, dy.p, N, O.P(cptr), N)
    assert np.array_equal(dy.download(), yu)
    # the first 200 rows only: the rest of y stays
    dy2 = ctx.array(np.full(N, 7.0))
    part = np.arange(201, dtype=np.int32)
    S.call("senk_sptrsv_csr_l_amc_f64", ctx.h, *(t.p for t in d[:3]), d[6].p, dy2.p, N, O.P(part), 200)
    out = dy2.download()
    assert np.array_equal(out[:200], yl[:200]) and np.all(out[200:] == 7.0)


def _bcsr(ctx, n, bnl, bnw, bsize, shuffle=False):
    """(device result of L, of U, oracle's of L, of U) on an elasticity (bnl 3) or 27-point system."""
    mat = S.gen_elasticity3(n, 2) if bnl == 3 else S.gen_convdiff27(n, 10.0)
    val, cind, rptr, N = S.padding(mat[2], mat[1], mat[0], bsize, len(mat[0]) - 1)
    sy = abmc_system(rptr, cind, val, bsize)
    fv, fc, fr = S.alloc_block_zero(sy["val"], sy["cind"], sy["rptr"], N, bnl, bnw)
    sp = S.split(oracle_ilu0(fv, fc, fr), fc, fr, N, "L-DU", True)
    bl, bu = S.csr2bcsr(*sp["L"], N, bnl, bnw), S.csr2bcsr(*sp["U"], N, bnl, bnw)
    x = np.random.default_rng(10).uniform(-1, 1, N)
    yl, yu = np.zeros(N), np.zeros(N)
    tail = (N, O.P(sy["cptr"]), sy["nc"], bsize, bnl, bnw)
    O.orc().or_sptrsv_bcsr_l_abmc_d(*(O.P(t) for t in bl), O.P(x), O.P(yl), *tail)
    O.orc().or_sptrsv_bcsr_u_abmc_d(*(O.P(t) for t in bu), O.P(yl), O.P(yu), *tail)
    if shuffle:  # the blocks of every row in another order (U keeps its diagonal ones first)
        rng, bs = np.random.default_rng(1), bnl * bnw
        for v, c, r, keep in ((*bl, 0), (*bu, bnl // bnw)):
            for g in range(N // bnl):
                k = np.arange(r[g] + keep, r[g + 1])
                o = rng.permutation(k)
                c[k], v.reshape(-1, bs)[k] = c[o].copy(), v.reshape(-1, bs)[o].copy()
    d = [ctx.array(t) for t in (*bl, *bu, x)]
    dy = ctx.zeros(N)
    S.call("senk_sptrsv_bcsr_l_abmc_f64", ctx.h, *(t.p for t in d[:3]), d[6].p, dy.p, *tail)
    t = dy.download()
    S.call("senk_sptrsv_bcsr_u_abmc_f64", ctx.h, *(t.p for t in d[3:6]), dy.p, dy.p, *tail)
    return t, dy.download(), yl, yu


# several blocks a wave, one, and blocks of more rows than a wave (in parts); every block shape
@pytest.mark.parametrize("bnl,bnw,bsize", [(1, 1, 5), (2, 1, 6), (2, 2, 64), (3, 1, 24), (3, 3, 24), (3, 3, 48),
                                           (3, 3, 63), (3, 3, 96), (4, 1, 20), (4, 2, 40), (4, 4, 128), (8, 1, 16),
                                           (8, 2, 8), (8, 4, 72), (8, 8, 64)])
def test_bcsr_abmc_bitwise(ctx, bnl, bnw, bsize):
    t, u, yl, yu = _bcsr(ctx, 9, bnl, bnw, bsize)
    assert np.array_equal(t, yl) and np.array_equal(u, yu)


@pytest.mark.parametrize("bnl,bnw,bsize", [(3, 3, 48), (2, 1, 8), (4, 4, 96)])
def test_bcsr_blocks_in_any_order(ctx, bnl, bnw, bsize):
    """Blocks of a row out of order: the same sums in another order (rows of at most 27 blocks,
    so a few tens of roundings each)."""
    t, u, yl, yu = _bcsr(ctx, 8, bnl, bnw, bsize, shuffle=True)
    assert relerr(t, yl) <= 1e-13 and relerr(u, yu) <= 1e-13


def _refused(ctx, bnl, bnw, n):
    """A block solve of n rows in a shape that no kernel takes: SENK_ERR_UNSUPPORTED (9)."""
    rptr = np.zeros(n // bnl + 1, np.int32)
    d = [ctx.array(t) for t in (np.zeros(1), np.zeros(1, np.int32), rptr, np.ones(n))]
    dy = ctx.zeros(n)
    cptr = np.array([0, 1], np.int32)
    assert S.lib().senk_sptrsv_bcsr_l_abmc_f64(ctx.h, *(t.p for t in d), dy.p, n, O.P(cptr), 1, n, bnl, bnw) == 9
    assert S.lib().senk_sptrsv_bcsr_u_abmc_f64(ctx.h, *(t.p for t in d), dy.p, n, O.P(cptr), 1, n, bnl, bnw) == 9


@pytest.mark.parametrize("bnl,bnw", [(5, 5), (6, 3), (6, 6), (16, 16)])
def test_a_refused_block_shape_leaves_the_next_solves_right(ctx, bnl, bnw):
    """The refusal neither uses nor turns over the vectors the solves share: before any other
    solve of a context, and between two solves of one size with different right-hand sides."""
    mats = [S.gen_vardiff7(8, s, 4.0, 1.5) for s in (3, 4)]
    with S.Context(0) as fresh:
        _refused(fresh, bnl, bnw, 240)
        _abmc_case(fresh, mats[0], 8, "connect", np.float64)
    for k in range(3):  # an odd and an even number of refusals between solves
        _abmc_case(ctx, mats[k & 1], 8, "connect", np.float64)
        for _ in range(k + 1):
            _refused(ctx, bnl, bnw, 480)
        _abmc_case(ctx, mats[(k + 1) & 1], 8, "connect", np.float64)
        _plan_case(ctx, mats[k & 1], np.float64)


def _gives_up(ctx, solve):
    """`solve` under a limit of one poll: its waits give up, and the context says so once."""
    assert S.lib().senk_ctx_set_trsv_polls(ctx.h, 1) == 0
    try:
        solve()
        return S.lib().senk_ctx_synchronize(ctx.h)
    finally:
        assert S.lib().senk_ctx_set_trsv_polls(ctx.h, 0) == 0


def _chain(ctx, n, dt=np.float64):
    """The L solve of a tridiagonal system on a plan (every row waits on the one before): a
    function that runs it, and its result's array and expected values."""
    rptr, cind, val = _tridiagonal(n)
    L, _ = (_typed(f, dt) for f in ilu_factors(dict(val=val, cind=cind, rptr=rptr)))
    x = np.random.default_rng(n).uniform(-1, 1, n).astype(dt)
    y = np.zeros_like(x)
    getattr(O.orc(), "or_sptrsv_l_" + ("d" if dt == np.float64 else "f"))(*(O.P(t) for t in L), O.P(x), O.P(y), n)
    plan = C.c_void_p()
    S.call("senk_trsv_plan_create", ctx.h, O.P(L[2]), O.P(L[1]), n, 0, C.byref(plan))
    d = [ctx.array(t) for t in (*L, x)]
    dy = ctx.zeros(n, dt)
    s = "f64" if dt == np.float64 else "f32"

    def run():
        S.call("senk_sptrsv_csr_l_" + s, ctx.h, plan, *(t.p for t in d), dy.p, n)

    return run, dy, y


@pytest.mark.parametrize("tickets", [0, 1])
@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_poll_limit(ctx, dt, tickets):
    run, dy, y = _chain(ctx, 500, dt)
    assert S.lib().senk_ctx_set_trsv_tickets(ctx.h, tickets) == 0
    try:
        for _ in range(2):
            assert _gives_up(ctx, run) == 11
            assert S.lib().senk_ctx_synchronize(ctx.h) == 0
            run()
            assert np.array_equal(dy.download(), y)
            run()
            assert np.array_equal(dy.download(), y)
    finally:
        S.lib().senk_ctx_set_trsv_tickets(ctx.h, -1)
    assert S.lib().senk_ctx_set_trsv_polls(ctx.h, -1) == 1


def test_a_wait_given_up_ends_only_its_own_solve(ctx):
    """The time-out word still set by an earlier solve (nothing has read it) does not end the
    waits of a later one, here of some 40 ms."""
    short, _, _ = _chain(ctx, 500)
    long, dy, y = _chain(ctx, 30000)
    assert S.lib().senk_ctx_set_trsv_polls(ctx.h, 1) == 0
    short()
    assert S.lib().senk_ctx_set_trsv_polls(ctx.h, 0) == 0
    long()
    assert S.lib().senk_ctx_synchronize(ctx.h) == 11  # the short one's
    assert np.array_equal(dy.download(), y)


def _abmc():
    rptr, cind, val = S.gen_vardiff7(20, 3, 4.0, 1.5)
    sy = abmc_system(rptr, cind, val, 8)
    sy["N"] = len(rptr) - 1
    sy["x"] = np.random.default_rng(8).uniform(-1, 1, sy["N"])
    return sy


def test_a_wait_given_up_is_reported_by_the_next_result(ctx):
    """Dot products and copies to the host, the sequential block form (which synchronises by
    itself) and a driver report it, once; the same calls are right again afterwards."""
    run, dy, y = _chain(ctx, 500)
    n, dot = len(y), C.c_double()
    buf = np.zeros(n)
    for read in (lambda: S.lib().senk_dot_f64(ctx.h, dy.p, dy.p, n, C.byref(dot)),
                 lambda: S.lib().senk_memcpy_dtoh(ctx.h, O.P(buf), dy.p, C.c_size_t(8 * n))):
        assert S.lib().senk_ctx_set_trsv_polls(ctx.h, 1) == 0
        run()
        assert read() == 11 and read() == 0
        assert S.lib().senk_ctx_set_trsv_polls(ctx.h, 0) == 0
    rptr, cind, val = _tridiagonal(200)
    L, _ = ilu_factors(dict(val=val, cind=cind, rptr=rptr))
    bl = S.csr2bcsr(*L, 200, 2, 2)
    d = [ctx.array(t) for t in (*bl, np.ones(200))]
    dz = ctx.zeros(200)
    seq = lambda: S.lib().senk_sptrsv_bcsr_l_f64(ctx.h, *(t.p for t in d), dz.p, 200, 2, 2)
    assert S.lib().senk_ctx_set_trsv_polls(ctx.h, 1) == 0
    assert seq() == 11
    assert S.lib().senk_ctx_set_trsv_polls(ctx.h, 0) == 0
    assert seq() == 0
    sy = _abmc()
    L, U = ilu_factors(sy)
    d = [ctx.array(t) for t in (sy["val"], sy["cind"], sy["rptr"], *L, *U, sy["x"])]
    dx, res = ctx.zeros(sy["N"]), S.senk_result()
    nrm_b = float(np.linalg.norm(sy["x"]))
    drv = lambda: S.lib().senk_abmc_ilu_gmresm_f64(ctx.h, *(t.p for t in d[:9]), O.P(sy["cptr"]), sy["nc"], 8, d[9].p,
                                                   dx.p, C.c_double(nrm_b), 100, 30, sy["N"], C.c_double(1e-8), 0,
                                                   C.byref(res), None, 0)
    assert S.lib().senk_ctx_set_trsv_polls(ctx.h, 1) == 0
    assert drv() == 11
    assert S.lib().senk_ctx_set_trsv_polls(ctx.h, 0) == 0
    dx.zero()
    assert drv() == 0 and res.converged == 1


@pytest.mark.parametrize("kind", ["ilu0", "ilub"])
def test_handles_without_the_sliced_layout_report_a_wait_given_up(ctx, kind):
    sy = _abmc()
    N = sy["N"]
    A, M = C.c_void_p(), C.c_void_p()
    S.call("senk_mat_create", ctx.h, N, O.P(sy["rptr"]), O.P(sy["cind"]), O.P(sy["val"]), 1, C.byref(A))
    opts = S.senk_ilu_opts(S.SENK_ILU0 if kind == "ilu0" else S.SENK_ILUB, 0, 2, 2, 1 << S.SENK_FACTOR_F64, 1)
    S.call("senk_prec_create_ilu", ctx.h, A, O.P(sy["rptr"]), O.P(sy["cind"]), O.P(sy["val"]), O.P(sy["cptr"]), sy["nc"],
           8, C.byref(opts), C.byref(M))
    db, dx, res = ctx.array(sy["x"]), ctx.zeros(N), S.senk_result()
    o = S.solve_opts(solver=S.SENK_GMRES, m=30, eps=1e-8, max_iter=3000)
    solve = lambda: S.lib().senk_solve(ctx.h, A, M, db.p, dx.p, C.byref(o), C.byref(res), None, 0)
    try:
        assert S.lib().senk_ctx_set_trsv_polls(ctx.h, 1) == 0
        S.call("senk_prec_apply_f64", M, db.p, dx.p)
        assert S.lib().senk_prec_check(M) == 11 and S.lib().senk_prec_check(M) == 0
        dx.zero()
        assert solve() == 11
        assert S.lib().senk_ctx_set_trsv_polls(ctx.h, 0) == 0
        dx.zero()
        assert solve() == 0 and res.converged == 1 and res.true_relres <= 1e-7
        assert S.lib().senk_prec_check(M) == 0
    finally:
        S.lib().senk_ctx_set_trsv_polls(ctx.h, 0)
        S.lib().senk_prec_destroy(M)
        S.lib().senk_mat_destroy(A)


@pytest.mark.parametrize("mode", [0, 1])
def test_tickets_by_number_and_by_arrival(ctx, mode):
    """Both ways of sharing out the rows give the sequential solve's bits, in any turn with the
    other (the counter's base moves with the launches that draw)."""
    assert S.lib().senk_ctx_set_trsv_tickets(ctx.h, 2) == 1
    try:
        for k, (bsize, dt) in enumerate([(1, np.float64), (8, np.float32), (64, np.float64)]):
            assert S.lib().senk_ctx_set_trsv_tickets(ctx.h, mode if k != 1 else 1 - mode) == 0
            _abmc_case(ctx, S.gen_convdiff27(11, 10.0), bsize, "connect", dt)
            _plan_case(ctx, S.gen_poisson7(9, 13, 5), dt)       # one XCD
            _plan_case(ctx, S.gen_poisson7(48, 46, 47), dt)     # all
            _plan_case(ctx, _tridiagonal(200), dt)
            _plan_case(ctx, _chain_then_wide(150, 150000), dt)
            t, u, yl, yu = _bcsr(ctx, 9, 3, 3, (24, 48, 96)[k])
            assert np.array_equal(t, yl) and np.array_equal(u, yu)
    finally:
        S.lib().senk_ctx_set_trsv_tickets(ctx.h, -1)


def test_solves_of_two_contexts_at_once(ctx):
    """Two contexts' solves in flight together, 8 streams of rows each, with neither waiting for
    the other on the host."""
    rptr, cind, val = S.gen_poisson7(48, 46, 47)
    N = len(rptr) - 1
    sy = abmc_system(rptr, cind, val, 1)
    L, U = ilu_factors(sy)
    x = np.random.default_rng(6).uniform(-1, 1, N)
    yl, yu = _seq(L, U, x)
    other = S.Context(0)
    try:
        runs = []
        for c in (ctx, other):
            d = [c.array(t) for t in (*L, *U, x)]
            plans = []
            for f, up in ((L, 0), (U, 1)):
                p = C.c_void_p()
                S.call("senk_trsv_plan_create", c.h, O.P(f[2]), O.P(f[1]), N, up, C.byref(p))
                plans.append(p)
            runs.append((c, d, plans, [c.zeros(N) for _ in range(2)]))
        for k in range(12):
            for c, d, plans, (a, b) in runs:
                if k % 3 == 2:
                    cp = O.P(sy["cptr"])
                    S.call("senk_sptrsv_csr_l_abmc_f64", c.h, *(t.p for t in d[:3]), d[6].p, a.p, N, cp, sy["nc"], 1)
                    S.call("senk_sptrsv_csr_u_abmc_f64", c.h, *(t.p for t in d[3:6]), a.p, b.p, N, cp, sy["nc"], 1)
                else:
                    S.call("senk_sptrsv_csr_l_f64", c.h, plans[0], *(t.p for t in d[:3]), d[6].p, a.p, N)
                    S.call("senk_sptrsv_csr_u_f64", c.h, plans[1], *(t.p for t in d[3:6]), a.p, b.p, N)
        for c, d, plans, (a, b) in runs:
            assert np.array_equal(a.download(), yl) and np.array_equal(b.download(), yu)
            for p in plans:
                S.lib().senk_trsv_plan_destroy(p)
        del runs, d, a, b
    finally:
        other.close()
