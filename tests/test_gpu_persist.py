"""The persistent solve and the launch-per-pass solve at the edges of their
shapes: rows around a workgroup's 1024 and around the row lengths of the
exchange, restarts around the tiers of eight basis vectors, 32 and 64, one
launch's largest row count and the first above it.

Bars: both forms give the same bits; the true FP64 residual by the oracle's
SpMV is at most 1e-10 (the solver's own stopping test, which it evaluates with
the same products)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import mke_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _line(n, width, seed):
    """Band matrix with `width` entries a row at most and a diagonal of 1.5
    times the sum of the row's others (at least 0.1), s: in the maximum norm
    the inverse is at most 1 / (0.5 s), and rounding the values to BF16 moves
    A by at most 2^-9 x 2.5 s, so a refinement step leaves at most 2.5 / 0.5 /
    2^9 = 1 % of the error beside its inner tolerance: every precision
    converges."""
    rng = np.random.default_rng(seed)
    half = width // 2
    offs = np.arange(-half, width - half)
    cols = np.arange(n)[:, None] + offs[None, :] * np.where(offs[None, :] == 0, 1, 3)
    there = (cols >= 0) & (cols < n)
    vals = rng.uniform(-1.0, 1.0, cols.shape)
    vals[:, offs == 0] = 0.0
    vals[:, offs == 0] = 1.5 * np.maximum(0.1, np.abs(vals).sum(1, keepdims=True))
    rp = np.concatenate([[0], np.cumsum(there.sum(1))]).astype(np.int32)
    return rp, cols[there].astype(np.int32), vals[there]


def _solve(A, b, **kw):
    x = torch.zeros_like(b)
    info = A.solve(x, b, rtol=1e-10, **kw)
    return x, info


def _check(n, width, **kw):
    csr = _line(n, width, n + width)
    A = P.Matrix.from_csr(n, n, *csr)
    bh = np.random.default_rng(n).standard_normal(n)
    b = torch.as_tensor(bh, device=DEV)
    x, info = _solve(A, b, persistent=True, **kw)
    y, ref = _solve(A, b, persistent=False, **kw)
    rel = np.linalg.norm(bh - O.spmv(*csr, x.cpu().numpy())) / np.linalg.norm(bh)
    assert info["converged"] and rel <= 1.001e-10, (info, rel)
    assert info["iterations"] == ref["iterations"] and torch.equal(x, y), (info, ref)
    here = n <= 262144 and kw.get("restart", 30) <= 32
    assert info["cycle_launches"] == (info["restarts"] if here else 0) and not ref["cycle_launches"]
    A.close()


@pytest.mark.parametrize("n", [1, 2, 63, 1023, 1024, 1025, 16384, 16385, 49153, 98305, 180225,
                               262144, 262145])
@pytest.mark.parametrize("ortho,precision", [(P.MGS, P.F64), (P.CGS2, P.F64), (P.MGS, P.F32),
                                             (P.CGS2, P.BF16)])
def test_persistent_and_passes_same_bits(n, ortho, precision):
    print("persistent n=%d ortho=%d precision=%d" % (n, ortho, precision), flush=True)
    _check(n, 5, ortho=ortho, precision=precision, restart=20)


@pytest.mark.parametrize("restart", [1, 2, 7, 8, 9, 16, 17, 24, 25, 31, 32, 33, 41, 64])
@pytest.mark.parametrize("ortho", [P.MGS, P.CGS2])
def test_restarts(restart, ortho):
    print("restart=%d ortho=%d" % (restart, ortho), flush=True)
    _check(3001, 8, ortho=ortho, restart=restart)
    _check(3001, 11, ortho=ortho, restart=restart)  # rows wider than the unrolled paths take


def test_start_vector_and_zero_right_side():
    print("start vector, zero right side", flush=True)
    n = 2500
    csr = _line(n, 6, 3)
    A = P.Matrix.from_csr(n, n, *csr)
    b = torch.as_tensor(np.random.default_rng(1).standard_normal(n), device=DEV)
    x0 = torch.as_tensor(np.random.default_rng(2).standard_normal(n), device=DEV)
    got = []
    for persistent in (True, False):
        x = x0.clone()
        info = A.solve(x, b, rtol=1e-10, use_x0=True, persistent=persistent)
        assert info["converged"]
        got.append(x)
        z = x0.clone()
        info = A.solve(z, torch.zeros_like(b), rtol=1e-10, persistent=persistent)
        assert info["converged"] and info["iterations"] == 0 and not z.any()
    assert torch.equal(got[0], got[1])
    A.close()


def _batch(A, B, x0=None, persistent=1, runs=None, **kw):
    """phg_gmres_batch with opts.persistent given; runs: whether the persistent
    form is the one that does."""
    import ctypes as C
    from mke_amd.phelm import GmresInfo, GmresOpts, check
    o = GmresOpts()
    P.lib().phg_gmres_default_opts(C.byref(o))
    o.rtol, o.persistent = 1e-10, persistent
    for k, v in kw.items():
        setattr(o, k, v)
    X = torch.zeros_like(B) if x0 is None else x0.clone()
    o.use_x0 = int(x0 is not None)
    infos = (GmresInfo * B.shape[1])()
    check(P.lib().phg_gmres_batch(A.h, B.shape[1], B.data_ptr(), X.data_ptr(), C.byref(o), infos,
                                  None), "phg_gmres_batch")
    runs = persistent if runs is None else runs
    assert all((i.cycle_launches > 0) == bool(runs) for i in infos)
    return X, [i.iterations for i in infos], [i.converged for i in infos]


@pytest.mark.parametrize("n,K", [(1, 3), (1000, 64), (1025, 1), (5000, 13), (40000, 7), (60000, 9),
                                 (262144, 2)])
@pytest.mark.parametrize("opts", [dict(ortho=P.CGS2), dict(ortho=P.CGS1, restart=8, diag_scale=1),
                                  dict(ortho=P.CGS1, precision=P.F32),
                                  dict(ortho=P.CGS2, precision=P.BF16, restart=17)])
def test_batch_persistent_and_launches(n, K, opts):
    """Column by column the persistent form reaches the residual that the
    launches reach, in as many steps up to one (their dots are added in other
    groups, so a residual at the stopping bound may fall on either side), a
    column's bits do not depend on the other columns, and with a start
    vector.  The last column is zero."""
    print("batch n=%d K=%d %s" % (n, K, opts), flush=True)
    csr = _line(n, 7, n + K)
    A = P.Matrix.from_csr(n, n, *csr)
    Bh = np.random.default_rng(n).standard_normal((n, K))
    if K > 1:
        Bh[:, -1] = 0.0
    B = torch.as_tensor(Bh, device=DEV)
    for x0 in (None, torch.as_tensor(np.random.default_rng(1).standard_normal((n, K)), device=DEV)):
        X, its, done = _batch(A, B, x0, 1, **opts)
        Y, ref, _ = _batch(A, B, x0, 0, **opts)
        assert all(done) and max(abs(a - b) for a, b in zip(its, ref)) <= 1, (its, ref)
        for q in range(K):
            x = np.ascontiguousarray(X[:, q].cpu().numpy())
            scale = np.linalg.norm(Bh[:, q]) or 1.0
            assert np.linalg.norm(Bh[:, q] - O.spmv(*csr, x)) <= 1.001e-10 * scale, q
        # both forms' errors are at most ||A^-1|| times the stopping residual,
        # and the diagonal is at least 3 x what the inverse's bound 1 / (0.5 s) needs
        assert float((X - Y).norm()) <= 1e-8 * max(1.0, float(Y.norm()))
        some = [0, K - 1] if K > 1 else [0]
        Z, _, _ = _batch(A, B[:, some].contiguous(), None if x0 is None else
                         x0[:, some].contiguous(), 1, **opts)
        for i, q in enumerate(some):
            assert torch.equal(Z[:, i], X[:, q]), q
    A.close()


@pytest.mark.parametrize("n", [255, 256, 257, 512, 513, 768, 769, 1280, 1281, 23553, 24833, 49000,
                               90113, 131072, 131073])
@pytest.mark.parametrize("precision", [P.F64, P.F32])
def test_half_workgroups_same_bits(n, precision):
    """Workgroups of 256 threads (up to 131,072 rows) at their edges: halves
    of a 1024-row block that are missing, partly filled or full, and the row
    lengths of the exchange.  Same bits as the launches, whose blocks are
    always whole."""
    _check(n, 7, ortho=P.MGS, precision=precision, restart=30)


@pytest.mark.parametrize("n,K", [(2304, 64), (2305, 64), (33000, 4)])
def test_half_and_whole_workgroups_same_column(n, K):
    """K columns take workgroups of 512 threads, two of them 256."""
    csr = _line(n, 7, n)
    A = P.Matrix.from_csr(n, n, *csr)
    B = torch.as_tensor(np.random.default_rng(n).standard_normal((n, K)), device=DEV)
    X, its, done = _batch(A, B, None, 1, ortho=P.CGS2)
    Z, some, _ = _batch(A, B[:, [0, K - 1]].contiguous(), None, 1, ortho=P.CGS2)
    assert all(done) and some == [its[0], its[-1]]
    assert torch.equal(Z, X[:, [0, K - 1]])
    A.close()


@pytest.mark.parametrize("polls", [1, 2, 4, 8, 16, 32])
def test_launches_that_do_not_start(polls, monkeypatch):
    """A limit of a few polls on a launch's first exchange makes launches give
    up, some or all of them: they are repeated, and the solve goes on as
    launches per pass when they keep failing.  The same bits and counts each
    time, with and without a start vector; batched columns reach their
    residual (the launches add their dots in other groups)."""
    print("start limit %d" % polls, flush=True)
    rng = np.random.default_rng(polls)
    for n, kw in ((700, dict(ortho=P.MGS)), (40000, dict(ortho=P.CGS2)),
                  (90000, dict(ortho=P.MGS, precision=P.F32)), (200000, dict(ortho=P.MGS))):
        csr = _line(n, 7, n)
        A = P.Matrix.from_csr(n, n, *csr)
        b = torch.as_tensor(rng.standard_normal(n), device=DEV)
        for x0 in (None, torch.as_tensor(rng.standard_normal(n), device=DEV)):
            got = []
            for limit in (None, polls):
                if limit:
                    monkeypatch.setenv("PHG_XCH_START", str(limit))
                x = torch.full_like(b, 7.0) if x0 is None else x0.clone()
                info = A.solve(x, b, rtol=1e-10, restart=4, use_x0=x0 is not None, **kw)
                monkeypatch.delenv("PHG_XCH_START", raising=False)
                got.append((x, info))
            (x, ref), (y, info) = got
            assert ref["restarts"] > 2 and ref["cycle_launches"] == ref["restarts"]
            keys = ("iterations", "restarts", "refinements", "rel_residual", "converged")
            assert all(info[k] == ref[k] for k in keys) and torch.equal(x, y), (n, info, ref)
            if polls == 1 and n == 200000:  # no workgroup but the last sees all slots at once
                assert info["cycle_launches"] == 16
        A.close()
    for n, K in ((1000, 40), (30000, 7)):
        csr = _line(n, 7, n)
        A = P.Matrix.from_csr(n, n, *csr)
        Bh = rng.standard_normal((n, K))
        Bh[:, -1] = 0.0
        B = torch.as_tensor(Bh, device=DEV)
        for x0 in (None, torch.as_tensor(rng.standard_normal((n, K)), device=DEV)):
            _, ref, _ = _batch(A, B, x0, 1, ortho=P.CGS2, restart=4)
            monkeypatch.setenv("PHG_XCH_START", str(polls))
            X, its, done = _batch(A, B, x0, 1, ortho=P.CGS2, restart=4)
            monkeypatch.delenv("PHG_XCH_START")
            assert all(done) and max(abs(a - c) for a, c in zip(its, ref)) <= 1, (its, ref)
            for q in range(K):
                x = np.ascontiguousarray(X[:, q].cpu().numpy())
                scale = np.linalg.norm(Bh[:, q]) or 1.0
                assert np.linalg.norm(Bh[:, q] - O.spmv(*csr, x)) <= 1.001e-10 * scale, q
        A.close()


def test_threads_solve_at_once():
    """Solves of several threads, each with a matrix and a stream of its own,
    small ones that run beside each other and ones that need the whole
    device: the bits of the same solve alone."""
    import threading
    print("threads", flush=True)
    sizes = [(3000, 1), (3000, 1), (20000, 2), (200000, 1), (60000, 4), (700, 30)]
    jobs = []
    for i, (n, K) in enumerate(sizes):
        A = P.Matrix.from_csr(n, n, *_line(n, 7, n + i))
        B = torch.as_tensor(np.random.default_rng(i).standard_normal((n, K)), device=DEV)
        X = torch.zeros_like(B)
        A.solve_batch(X, B, rtol=1e-10)
        jobs.append((A, B, X))
    torch.cuda.synchronize()
    bad, gate = [], threading.Barrier(len(jobs))

    def work(i):
        A, B, X = jobs[i]
        try:
            stream = torch.cuda.Stream()
            gate.wait(60)
            with torch.cuda.stream(stream):
                for _ in range(40):
                    Y = torch.zeros_like(B)
                    A.solve_batch(Y, B, rtol=1e-10, stream=stream)
                    if not torch.equal(X, Y):
                        bad.append(i)
        except Exception as e:  # reported below: an assertion here would be lost
            bad.append((i, e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad


@pytest.mark.parametrize("n,opts,inside,outside", [
    (163841, dict(ortho=P.CGS1, precision=P.F32), 11, 13),
    (40961, dict(ortho=P.CGS1, restart=8, diag_scale=1), 24, 32),
    (40961, dict(ortho=P.CGS1, restart=8, diag_scale=1), 40, 48)])
def test_batch_widths_of_both_forms(n, opts, inside, outside):
    """Numbers of columns with the same padded width on either side of the
    line between the forms: a column's bits are the same for every number on
    one side, and across the line the residual is."""
    csr = _line(n, 7, n)
    A = P.Matrix.from_csr(n, n, *csr)
    Bh = np.random.default_rng(n).standard_normal((n, outside + 1))
    B = torch.as_tensor(Bh, device=DEV)

    def run(k, runs):
        X, its, done = _batch(A, B[:, :k].contiguous(), None, 1, runs=runs, **opts)
        assert all(done)
        x = np.ascontiguousarray(X[:, 1].cpu().numpy())
        assert np.linalg.norm(Bh[:, 1] - O.spmv(*csr, x)) <= 1.001e-10 * np.linalg.norm(Bh[:, 1])
        return X[:, :2], its[:2]

    few, most, over = run(2, True), run(inside, True), run(outside, False)
    assert torch.equal(few[0], most[0]) and few[1] == most[1]
    if outside == 13:
        assert torch.equal(over[0], run(outside + 1, False)[0])
    assert max(abs(a - b) for a, b in zip(most[1], over[1])) <= 1


def test_batch_of_more_than_one_launch():
    """A launch ends after 4,096 Arnoldi steps of a column; slow columns take
    several, beside columns that stop in the first."""
    nx = 140
    i = np.arange(nx * nx)
    x, y = i % nx, i // nx
    cols = np.stack([i - nx, i - 1, i, i + 1, i + nx], 1)
    there = np.stack([y > 0, x > 0, x >= 0, x < nx - 1, y < nx - 1], 1)
    vals = np.full(cols.shape, -1.0)
    vals[:, 2] = 4.0 + 1e-4
    csr = (np.concatenate([[0], np.cumsum(there.sum(1))]).astype(np.int32),
           cols[there].astype(np.int32), vals[there])
    n = nx * nx
    A = P.Matrix.from_csr(n, n, *csr)
    Bh = np.random.default_rng(5).standard_normal((n, 3))
    Bh[:, 1] = O.spmv(*csr, np.sin(np.pi * (x + 1) / (nx + 1)) * np.sin(np.pi * (y + 1) / (nx + 1)))
    B = torch.as_tensor(Bh, device=DEV)
    X, its, done = _batch(A, B, None, 1, ortho=P.CGS2, restart=8)
    Y, ref, _ = _batch(A, B, None, 0, ortho=P.CGS2, restart=8)
    print(its, ref)
    assert all(done) and its[0] > 4096 and its[1] < 10, its
    for q in range(3):
        r = Bh[:, q] - O.spmv(*csr, np.ascontiguousarray(X[:, q].cpu().numpy()))
        assert np.linalg.norm(r) <= 1.001e-10 * np.linalg.norm(Bh[:, q]), q
    # the same stopping residual: errors of at most cond(A) = 8 / 0.0011 times it
    assert float((X - Y).norm()) <= 2 * 7400 * 1e-10 * float(Y.norm())


def test_batch_with_columns_that_are_not_finite():
    """Columns with a NaN or an infinity stop at once and leave the others'
    bits alone."""
    n, K = 20000, 5
    csr = _line(n, 7, n)
    A = P.Matrix.from_csr(n, n, *csr)
    B = torch.as_tensor(np.random.default_rng(8).standard_normal((n, K)), device=DEV)
    X, its, _ = _batch(A, B, None, 1, ortho=P.CGS2)
    B[17, 1], B[n - 1, 3] = float("nan"), float("inf")
    for persistent in (1, 0):
        Y, got, done = _batch(A, B, None, persistent, ortho=P.CGS2)
        assert [bool(d) for d in done] == [True, False, True, False, True]
        assert got[1] == 0 and got[3] == 0 and abs(got[0] - its[0]) <= 1
        if persistent:
            assert torch.equal(Y[:, ::2], X[:, ::2])
    Z, got, done = _batch(A, B[:, ::2].contiguous(), None, 1, ortho=P.CGS2)
    assert all(done) and torch.equal(Z, X[:, ::2])


@pytest.mark.parametrize("width", [8, 9, 15, 16, 17, 27])
def test_rows_wider_than_one_group(width):
    """Rows around multiples of the eight entries that are loaded together,
    in both forms of the single and the batched solve and each precision
    (ragged at the ends of the band)."""
    n = 2600
    for ortho, precision in ((P.MGS, P.F64), (P.CGS2, P.F32), (P.MGS, P.BF16)):
        _check(n, width, ortho=ortho, precision=precision)
    csr = _line(n, width, width)
    A = P.Matrix.from_csr(n, n, *csr)
    Bh = np.random.default_rng(width).standard_normal((n, 5))
    B = torch.as_tensor(Bh, device=DEV)
    for opts in (dict(ortho=P.CGS2), dict(ortho=P.CGS1, precision=P.F32),
                 dict(ortho=P.CGS2, precision=P.BF16)):
        its = []
        for persistent in (1, 0):
            X, i, done = _batch(A, B, None, persistent, **opts)
            its.append(i)
            assert all(done)
            for q in range(5):
                r = Bh[:, q] - O.spmv(*csr, np.ascontiguousarray(X[:, q].cpu().numpy()))
                assert np.linalg.norm(r) <= 1.001e-10 * np.linalg.norm(Bh[:, q])
        assert max(abs(a - b) for a, b in zip(*its)) <= 1, its
    A.close()
