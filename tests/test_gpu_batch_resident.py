"""The resident batch kernel (a team of workgroups per system, systems in rounds) against the CPU oracle, bit for bit,
where its teams and rounds can go wrong."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(gpu, orc, systems, tol=0.0, max_iter=6, guard=0, bad=()):
    srp, rp, col, val = gpu.block_diag(systems)
    n = int(srp[-1])
    b = gpu.uniform(5, 0, n) - 0.5
    x0 = b / 20  # better than zero: all eigenvalues lie in (0, 20)
    for s in bad:  # guesses far worse than zero
        x0[srp[s]:srp[s + 1]] = 1e3
    p = gpu.cg_params(method=gpu.CG_PIPELINED, tol=tol, max_iter=max_iter, x0_guard=guard)
    with gpu.CgBatchPlan(srp, rp, col, val, p) as plan:
        plan.set_rhs(b)
        plan.set_x0(x0)
        for _ in range(2):  # the second solve starts over
            _, iters, _, hist, t = plan.solve(hist_cap=max_iter + 1)
            x = plan.x()
        rejected = plan.x0_rejected()
    for s, (r, c, v) in enumerate(systems):
        sl = slice(srp[s], srp[s + 1])
        start = np.zeros(sl.stop - sl.start) if s in bad and guard else x0[sl]
        _, ox, ohist, oit = orc.cg(orc.Csr(r, c, v), b[sl], x0=start, tol=tol, max_iter=max_iter, variant="pipelined")
        assert iters[s] == oit and rejected[s] == (1 if guard and s in bad else 0)
        assert np.array_equal(x[sl], ox) and np.array_equal(hist[s, :oit + 1], ohist)
    return t


def test_batch_resident_sizes(gpu, orc):
    """One row, one chunk and one row more, rows of 3 and of 7 entries, in one round."""
    systems = [gpu.tridiag(n, 1 + n) for n in (2, 63, 1024, 1025, 2047, 5000)]
    t = _check(gpu, orc, systems)
    assert t["block_threads"] == 256
    _check(gpu, orc, systems + [gpu.poisson3d(9, 10, 11), gpu.poisson3d(1, 1, 1), gpu.poisson3d(16, 16, 16)])


def test_batch_resident_rounds(gpu, orc):
    """More chunks than workgroups: teams of several rounds, one of them as large as half the chip."""
    systems = [gpu.poisson3d(8 + i % 7, 20, 30) for i in range(60)] + [gpu.poisson3d(64, 64, 64)] * 3
    _check(gpu, orc, systems, tol=1e-6, max_iter=400)


def test_batch_resident_largest_system(gpu, orc):
    """A system of exactly 512 chunks, and one chunk more (the general kernel's)."""
    small = gpu.tridiag(3000, 4)
    t = _check(gpu, orc, [small, gpu.tridiag(524288, 3), small])
    assert t["block_threads"] == 256
    t = _check(gpu, orc, [small, gpu.tridiag(1048577, 3)])
    assert t["block_threads"] == 1024


@pytest.mark.parametrize("tol,max_iter", [(1e-7, 200), (0.0, 3)])
def test_batch_resident_guard(gpu, orc, tol, max_iter):
    systems = [gpu.poisson3d(10, 11, 12), gpu.poisson3d(20, 9, 14), gpu.tridiag(4000, 9)]
    _check(gpu, orc, systems, tol=tol, max_iter=max_iter, guard=1, bad=(1,))


def _line(n):
    """The 1D Laplacian (about n iterations to converge)."""
    col = (np.arange(n)[:, None] + np.arange(-1, 2)).astype(np.int32)
    ok = (col >= 0) & (col < n)
    rp = np.zeros(n + 1, dtype=np.int32)
    rp[1:] = np.cumsum(ok.sum(1))
    return rp, col[ok], np.broadcast_to([-1.0, 2.0, -1.0], col.shape)[ok]


def test_batch_resident_waits_for_longer_systems(gpu):
    """A team of the second round whose members come from a system of the first round that ends at once and from one
    that iterates for many times the watchdog's limit waits for the latter, and solves its system as a solve alone does."""
    chunks = (260, 250, 240, 230, 225)  # rounds {260, 250, 240} and {230, 225}; the last spans the first two
    max_iter, limit_us = 3000, 2000
    systems = [_line(1024 * c) for c in chunks]
    srp, rp, col, val = gpu.block_diag(systems)
    b = gpu.uniform(8, 0, int(srp[-1])) - 0.5
    b[srp[1]:srp[4]] = 0.0  # solved by x0 = 0
    p = gpu.cg_params(method=gpu.CG_PIPELINED, tol=1e-8, max_iter=max_iter, spin_limit_us=limit_us)
    with gpu.CgBatchPlan(srp, rp, col, val, p) as plan:
        plan.set_rhs(b)
        plan.set_x0(None)
        st, iters, stat, _, t = plan.solve()
        x = plan.x()
    assert t["block_threads"] == 256 and t["kernel_ms"] > 5e-3 * limit_us
    assert st == gpu.ENOTCONV and list(iters) == [max_iter, 0, 0, 0, max_iter]
    for s in (0, 4):
        alone = gpu.cg(*systems[s], b[srp[s]:srp[s + 1]], method=gpu.CG_PIPELINED, tol=1e-8, max_iter=max_iter)
        assert alone[0] == gpu.ENOTCONV and np.array_equal(x[srp[s]:srp[s + 1]], alone[1])


def test_batch_tune_cache_names_the_candidates(gpu, tmp_path):
    """A winner is only looked up by plans that choose among the same candidates: not one from a plan that has no
    resident kernel, nor one of a file from before there was one."""
    systems = [gpu.poisson3d(8, 9, 10), gpu.poisson3d(20, 9, 14)]
    srp, rp, col, val = gpu.block_diag(systems)
    b = gpu.uniform(5, 0, int(srp[-1]))
    cache = tmp_path / "tune.txt"

    def tune(**kw):
        p = gpu.cg_params(method=gpu.CG_PIPELINED, tol=1e-8, max_iter=500, **kw)
        with gpu.CgBatchPlan(srp, rp, col, val, p) as plan:
            plan.set_rhs(b)
            plan.set_x0(None)
            first = plan.resident()
            won = plan.tune(trial_iters=5, cache_path=str(cache))
            return first, won, plan.resident(), len(cache.read_text().splitlines())

    first, won, resident, lines = tune(block_threads=1024)
    assert not first and not resident and lines == 1
    first, won, resident, lines = tune()
    assert first and lines == 2
    assert tune() == (True, won, resident, 2)  # its own line is found again
    # a line as it was written before there was a resident kernel
    old = cache.read_text().splitlines()[1].split()[0].split("|format=")[0]
    cache.write_text(f"{old} 4 256 0\n")
    assert tune()[3] == 2


def test_batch_resident_single_chunks_come_last(gpu):
    """Systems of one chunk, whose workgroups have no barriers that a later team could see them pass, iterate for a
    multiple of the watchdog's limit beside systems that take two rounds of almost the whole grid."""
    limit_us = 1000
    systems = [_line(1024 * c) for c in (700, 750)] + [_line(1000 + i) for i in range(60)]
    srp, rp, col, val = gpu.block_diag(systems)
    b = gpu.uniform(9, 0, int(srp[-1])) - 0.5
    b[:srp[2]] = 0.0  # the large ones are solved by x0 = 0
    p = gpu.cg_params(method=gpu.CG_PIPELINED, tol=1e-8, max_iter=3000, spin_limit_us=limit_us)
    with gpu.CgBatchPlan(srp, rp, col, val, p) as plan:
        plan.set_rhs(b)
        plan.set_x0(None)
        st, iters, stat, _, t = plan.solve()
        x = plan.x()
        assert plan.resident() and t["kernel_ms"] > 2e-3 * limit_us
    assert list(iters[:2]) == [0, 0] and not x[:srp[2]].any()
    for s in (2, 30, 61):
        alone = gpu.cg(*systems[s], b[srp[s]:srp[s + 1]], method=gpu.CG_PIPELINED, tol=1e-8, max_iter=3000)
        assert stat[s] == alone[0] and iters[s] == alone[3] and np.array_equal(x[srp[s]:srp[s + 1]], alone[1])
