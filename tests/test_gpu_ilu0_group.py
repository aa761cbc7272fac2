"""The grouped ILU(0) kernel (several lanes per row, rows in LDS) against the oracle's Ilu0.

Same operations per entry in the same order: the same bits in FP64 and FP32, for every block
size it takes, rows around its two group widths, and the cases it hands on."""
import numpy as np
import pytest

import senk_amd as S
from oracle import oracle as O
from tests.helpers import abmc_system

pytestmark = pytest.mark.gpu


def _factor(ctx, val, cind, rptr, N, dt, cptr=None, nc=0, bsize=1):
    v = np.ascontiguousarray(val.astype(dt))
    fo = v.copy()
    assert getattr(O.orc(), "or_ilu0_d" if dt == np.float64 else "or_ilu0_f")(O.P(fo), O.P(cind), O.P(rptr), N) == 0
    d = [ctx.array(t) for t in (v, cind, rptr)]
    S.call("senk_ilu0_f64" if dt == np.float64 else "senk_ilu0_f32", ctx.h, *(t.p for t in d), N,
           None if cptr is None else O.P(cptr), nc, bsize, O.P(rptr), O.P(cind))
    return d[0].download(), fo


@pytest.mark.parametrize("bsize", [1, 2, 4, 8, 16, 32, 64, 48])
@pytest.mark.parametrize("gen", ["poisson7", "convdiff27", "unstructured"])
@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_colored_bitwise(ctx, bsize, gen, dt):
    mat = {"poisson7": lambda: S.gen_poisson7(11, 9, 7), "convdiff27": lambda: S.gen_convdiff27(8, 10.0),
           "unstructured": lambda: S.gen_unstructured(1500, 4)}[gen]()
    val, cind, rptr, N = S.padding(mat[2], mat[1], mat[0], bsize, len(mat[0]) - 1)
    sy = abmc_system(rptr, cind, val, bsize)
    f, fo = _factor(ctx, sy["val"], sy["cind"], sy["rptr"], N, dt, sy["cptr"], sy["nc"], bsize)
    assert np.array_equal(f, fo)


# dependency levels (lists of rows), up to 16 entries a row, 17, and up to 225
@pytest.mark.parametrize("width", [7, 16, 17, 90, 400])
@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_levels_of_banded_rows_bitwise(ctx, width, dt):
    rng, N, h = np.random.default_rng(width), 700, width // 2
    rows = [np.unique(np.clip(np.concatenate([[i], i + rng.integers(-3 * h, 3 * h + 1, width - 1)]), 0, N - 1))
            for i in range(N)]
    rptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    cind = np.concatenate(rows).astype(np.int32)
    val = rng.uniform(-1, 1, len(cind))
    for i in range(N):
        val[rptr[i] + np.searchsorted(rows[i], i)] = 2.0 + len(rows[i])
    f, fo = _factor(ctx, val, cind, rptr, N, dt)
    assert np.array_equal(f, fo)


def _rows_of(N, width, seed):
    """Rows of exactly `width` ascending columns, near the diagonal, which is among them."""
    rng, out = np.random.default_rng(seed), []
    for i in range(N):
        lo = min(max(0, i - width), N - 2 * width)
        c = rng.choice(np.setdiff1d(np.arange(lo, lo + 2 * width), [i]), width - 1, replace=False)
        out.append(np.sort(np.append(c, i)))
    rptr = (np.arange(N + 1) * width).astype(np.int32)
    cind = np.concatenate(out).astype(np.int32)
    val = rng.uniform(-1, 1, len(cind))
    val[cind == np.repeat(np.arange(N), width)] = 2.0 + width
    return rptr, cind, val


# The grouped kernel holds up to 64 KB of entries (12 bytes in FP64, 8 in FP32) per workgroup of
# 16 rows, or of 64 in blocks of 64: the longest rows it takes and the shortest it hands on.
@pytest.mark.parametrize("bsize,dt,width", [(1, np.float64, 341), (1, np.float64, 342), (1, np.float32, 512),
                                            (1, np.float32, 513), (8, np.float64, 341), (8, np.float64, 342),
                                            (64, np.float64, 85), (64, np.float64, 86), (64, np.float32, 128),
                                            (64, np.float32, 129)])
def test_rows_around_the_lds_limit_bitwise(ctx, bsize, dt, width):
    N = 1152
    rptr, cind, val = _rows_of(N, width, width)
    if bsize == 1:  # dependency levels
        f, fo = _factor(ctx, val, cind, rptr, N, dt)
    else:
        sy = abmc_system(rptr, cind, val, bsize)
        f, fo = _factor(ctx, sy["val"], sy["cind"], sy["rptr"], N, dt, sy["cptr"], sy["nc"], bsize)
    assert np.array_equal(f, fo)


@pytest.mark.parametrize("where", ["block", "other"])
def test_zero_pivot_inside_and_outside_the_block(ctx, where):
    N, bs = 8, 4
    A = np.eye(N) * 3
    i, j = (1, 0) if where == "block" else (5, 2)
    A[i, j], A[j, j] = 1.0, 0.0
    rptr, cind, val = [0], [], []
    for r in range(N):
        for c in range(N):
            if A[r, c] != 0 or r == c:
                cind.append(c)
                val.append(A[r, c])
        rptr.append(len(cind))
    d = [ctx.array(np.array(t, dt)) for t, dt in ((val, np.float64), (cind, np.int32), (rptr, np.int32))]
    cptr = np.array([0, 1, 2], np.int32)
    assert S.lib().senk_ilu0_f64(ctx.h, *(t.p for t in d), N, O.P(cptr), 2, bs, None, None) == 3


def _elimination(val, cind, rptr, N):
    """ILU(0) by columns, whatever the order of a row's later entries: every entry gets its updates
    in increasing pivot column."""
    v, at = val.copy(), [dict(zip(cind[rptr[i]:rptr[i + 1]].tolist(), range(rptr[i], rptr[i + 1]))) for i in range(N)]
    for i in range(N):
        for k in sorted(c for c in at[i] if c < i):
            l = v[at[i][k]] / v[at[k][k]]
            v[at[i][k]] = l
            for c, q in at[i].items():
                if c > k and c in at[k]:
                    v[q] -= l * v[at[k][c]]
    return v


@pytest.mark.parametrize("order", ["ascending", "shuffled"])
def test_rows_whose_later_entries_are_in_any_order(ctx, order):
    """Entries beyond the diagonal out of order, in rows that no other row eliminates with."""
    rng, h = np.random.default_rng(3), 48
    N, rows = 2 * h, []
    for i in range(N):
        up = np.arange(i + 1, N)
        up = np.sort(rng.choice(up, min(len(up), 14), replace=False))
        if i >= h and order == "shuffled":
            up = rng.permutation(up)
        low = np.sort(rng.choice(min(i, h), min(i, h, 9), replace=False)) if i else np.zeros(0, int)
        rows.append(np.concatenate([low, [i], up]))
    rptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    cind = np.concatenate(rows).astype(np.int32)
    val = rng.uniform(-1, 1, len(cind))
    for i in range(N):
        val[rptr[i] + np.flatnonzero(rows[i] == i)[0]] = 20.0
    d = [ctx.array(t) for t in (val, cind, rptr)]
    S.call("senk_ilu0_f64", ctx.h, *(t.p for t in d), N, None, 0, 1, O.P(rptr), O.P(cind))
    assert np.array_equal(d[0].download(), _elimination(val, cind, rptr, N))
