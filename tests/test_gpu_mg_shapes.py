"""The V-cycle's launches at the shapes they change with: one level above
the direct solve, several, up to eight columns (fused passes) and more.

Bar: applied twice to the same right-hand sides in other batch widths, a
solve reaches the residual it stops at, and its solutions differ by at most
what two residuals of 1e-10 allow (the Helmholtz operator here is
conditioned well enough for a forward error of 1e-8)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import mke_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("precision", [P.F64, P.F32])
@pytest.mark.parametrize("level,widths", [(1, (1, 3)), (2, (1, 9)), (3, (1, 2, 8, 9)),
                                          (4, (1, 5, 16)), (5, (1, 8, 17, 64)), (6, (1, 8, 33))])
def test_vcycle_shapes(level, widths, precision):
    print("mg level=%d widths=%s precision=%d" % (level, widths, precision), flush=True)
    pm = P.Mesh.sphere(level)
    cm, cl = P.helmholtz_coeffs(tau=1.0, sigma=0.0, theta=1.0, mu=1e-2)
    mg = P.Multigrid(pm, P.HELMHOLTZ, cm, cl)
    csr = mg.A.csr()
    n = pm.inner_size
    Bh = np.random.default_rng(level).standard_normal((n, max(widths)))
    B = torch.as_tensor(Bh, device=DEV)
    first = None
    for k in widths:
        X = torch.zeros((n, k), dtype=torch.float64, device=DEV)
        infos = mg.solve_batch(X, B[:, :k].contiguous(), rtol=1e-10, precision=precision)
        x = X.cpu().numpy()
        for q in range(k):
            rel = np.linalg.norm(Bh[:, q] - O.spmv(*csr, np.ascontiguousarray(x[:, q])))
            assert infos[q]["converged"] and rel <= 1.001e-10 * np.linalg.norm(Bh[:, q]), (k, q)
        if first is None:
            first = x[:, 0]
        assert np.linalg.norm(x[:, 0] - first) <= 1e-8 * np.linalg.norm(first), k


def test_graph_serves_other_arrays():
    """The captured cycle does not depend on the caller's arrays: solves into
    changing buffers give the bits of a fresh object's first solve."""
    pm = P.Mesh.sphere(4)
    mg = P.Multigrid(pm, P.LAPLACE)
    n = pm.inner_size
    B = [torch.as_tensor(np.random.default_rng(s).standard_normal((n, 2)), device=DEV)
         for s in range(3)]
    got = []
    for _ in range(2):
        for b in B:
            X = torch.zeros_like(b)
            mg.solve_batch(X, b.clone(), rtol=1e-10)
            got.append(X)
    for k, b in enumerate(B):
        fresh = P.Multigrid(pm, P.LAPLACE)
        X = torch.zeros_like(b)
        fresh.solve_batch(X, b, rtol=1e-10)
        assert torch.equal(X, got[k]) and torch.equal(X, got[k + 3])
