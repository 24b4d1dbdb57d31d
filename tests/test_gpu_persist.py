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
