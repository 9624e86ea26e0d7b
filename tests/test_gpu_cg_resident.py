"""Resident CG kernels (vectors, and for smaller systems the matrix, in registers for the whole solve)
against the CPU oracle, bit for bit, at the sizes where one kernel gives way to the next."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

METHODS = {"standard": 0, "pipelined": 1, "ir": 2}


def _check(gpu, orc, rp, col, val, method, iters, fmt=0, seed=3):
    n = rp.size - 1
    b = gpu.uniform(seed, 0, n) - 0.5
    x0 = gpu.uniform(seed, 1, n) - 0.5
    A = orc.Csr(rp, col, val)
    if method == "ir":
        kw = dict(tol=1e-9, max_outer=2, inner_tol=1e-3)
        p = gpu.cg_params(method=2, max_iter=iters, matrix_format=fmt, **kw)
    else:
        p = gpu.cg_params(method=METHODS[method], tol=0.0, max_iter=iters, matrix_format=fmt)
    with gpu.CgPlan(rp, col, val, p) as plan:
        plan.set_rhs(b)
        plan.set_x0(x0)
        for _ in range(2):  # a second solve on the same plan starts over
            st, hist, it, t = plan.solve()
            x = plan.x()
            if method == "ir":
                ost, ox, ohist, oouter, oit = orc.cg_ir(A, b, x0=x0, inner_max=iters, **kw)
                assert t["outer_iterations"] == oouter
            else:
                ost, ox, ohist, oit = orc.cg(A, b, x0=x0, tol=0.0, max_iter=iters, variant=method)
            assert it == oit and st == ost
            assert np.array_equal(x, ox) and np.array_equal(hist, ohist)


# rows: one, one chunk, a ragged last chunk, as many chunks as CUs and one more, twice as many and
# more, four times and more, eight times and more (where the general kernel takes over)
@pytest.mark.parametrize("method", list(METHODS))
@pytest.mark.parametrize("dims", [(1, 1, 1), (16, 8, 8), (31, 7, 5), (64, 64, 64), (64, 64, 65), (128, 64, 64),
                                  (128, 64, 65), (128, 128, 64), (128, 127, 65), (128, 128, 128), (128, 128, 129)])
def test_resident_poisson(gpu, orc, dims, method):
    _check(gpu, orc, *gpu.poisson3d(*dims), method, 4)


@pytest.mark.parametrize("method", list(METHODS))
@pytest.mark.parametrize("n", [5, 1025, 262145, 524289, 1048577])
def test_resident_tridiagonal(gpu, orc, n, method):
    _check(gpu, orc, *gpu.tridiag(n, 2), method, 4)


@pytest.mark.parametrize("method", list(METHODS))
@pytest.mark.parametrize("dims,fmt", [((128, 64, 65), 2), ((128, 128, 65), 2), ((128, 128, 65), 1)])
def test_resident_asked_formats(gpu, orc, dims, fmt, method):
    _check(gpu, orc, *gpu.poisson3d(*dims), method, 4, fmt)


def _banded(n, half, seed):
    """Symmetric, strictly diagonally dominant, 2*half + 1 entries a row."""
    rng = np.random.default_rng(seed)
    bands = [rng.uniform(-1, 0, n) for _ in range(half)]
    rows = []
    for r in range(n):
        lo = [(r - k, bands[k - 1][r - k]) for k in range(half, 0, -1) if r - k >= 0]
        hi = [(r + k, bands[k - 1][r]) for k in range(1, half + 1) if r + k < n]
        rows.append(lo + [(r, 2.0 * half + 1.0)] + hi)
    rp = np.zeros(n + 1, dtype=np.int32)
    rp[1:] = np.cumsum([len(r) for r in rows])
    return (rp, np.array([c for r in rows for c, _ in r], dtype=np.int32), np.array([v for r in rows for _, v in r]))


@pytest.mark.parametrize("method", list(METHODS))
@pytest.mark.parametrize("half", [0, 2, 3, 4])
def test_resident_row_widths(gpu, orc, half, method):
    """1, 5, 7 and 9 entries a row (the last too wide for the registers)."""
    _check(gpu, orc, *_banded(2500, half, half), method, 9)


def _nine_diagonals(n):
    """Nine full diagonals but for the pair of entries (10, 11) and (11, 10), which a diagonal's storage holds as zeros."""
    offs = np.array([-900, -3, -2, -1, 0, 1, 2, 3, 900])
    col = (np.arange(n)[:, None] + offs).astype(np.int32)
    ok = (col >= 0) & (col < n)
    ok[10, 5] = ok[11, 3] = False
    rp = np.zeros(n + 1, dtype=np.int32)
    rp[1:] = np.cumsum(ok.sum(1))
    return rp, col[ok], np.broadcast_to(np.where(offs == 0, 10.0, -1.0), col.shape)[ok]


@pytest.mark.parametrize("method", ["standard", "pipelined"])
def test_nine_diagonals_below_2_20_rows_keep_sell(gpu, orc, method):
    """Stored by rows, an infinite guess reaches only the rows that hold its column: <r, r> is infinite, not NaN (an
    infinity times a diagonal's stored zero)."""
    rp, col, val = _nine_diagonals(700000)
    b = gpu.uniform(3, 0, 700000) - 0.5
    x0 = np.zeros(700000)
    x0[11] = np.inf
    A = orc.Csr(rp, col, val)
    ost, ox, ohist, oit = orc.cg(A, b, x0=x0, tol=1e-8, max_iter=3, variant=method)
    st, x, hist, it, t = gpu.cg(rp, col, val, b, x0=x0, method=METHODS[method], tol=1e-8, max_iter=3)
    assert np.isinf(ohist[0]) and np.isinf(hist[0])
    assert (st, it) == (ost, oit) and np.array_equal(x, ox)
    _check(gpu, orc, rp, col, val, method, 3)


def _pairs(n, seed):
    """Rows of up to 4 entries at random columns (no diagonals to store them by)."""
    rng = np.random.default_rng(seed)
    rows = [np.arange(n)]
    cols = [np.arange(n)]
    for _ in range(3):
        p = rng.permutation(n)[: n // 2 * 2].reshape(-1, 2)
        rows += [p[:, 0], p[:, 1]]
        cols += [p[:, 1], p[:, 0]]
    r, c = np.concatenate(rows), np.concatenate(cols)
    key = np.unique(r * np.int64(n) + c)
    r, c = key // n, key % n
    rp = np.zeros(n + 1, dtype=np.int32)
    rp[1:] = np.cumsum(np.bincount(r, minlength=n))
    return rp, c.astype(np.int32), np.where(r == c, 4.0, -1.0)


@pytest.mark.parametrize("method", list(METHODS))
@pytest.mark.parametrize("matrix", ["poisson", "pairs"])
def test_streamed_infinite_guess(gpu, orc, matrix, method):
    """An infinity in the guess reaches the rows that hold its column and no others, as in the oracle: <r, r> is
    infinite, not NaN."""
    rp, col, val = gpu.poisson3d(96, 96, 60) if matrix == "poisson" else _pairs(540000, 5)
    n = rp.size - 1
    assert n > 2 ** 19
    b = gpu.uniform(3, 0, n) - 0.5
    for at in (0, 95):
        x0 = np.zeros(n)
        x0[at] = np.inf
        A = orc.Csr(rp, col, val)
        if method == "ir":
            ost, ox, ohist, _, oit = orc.cg_ir(A, b, x0=x0, tol=1e-9, inner_max=5, max_outer=2, inner_tol=1e-3)
            kw = dict(tol=1e-9, max_iter=5, max_outer=2, inner_tol=1e-3)
        else:
            ost, ox, ohist, oit = orc.cg(A, b, x0=x0, tol=1e-8, max_iter=3, variant=method)
            kw = dict(tol=1e-8, max_iter=3)
        st, x, hist, it, _ = gpu.cg(rp, col, val, b, x0=x0, method=METHODS[method], **kw)
        assert np.isinf(ohist[0]) and np.isinf(hist[0])
        assert (st, it) == (ost, oit) and np.array_equal(x, ox, equal_nan=True)
