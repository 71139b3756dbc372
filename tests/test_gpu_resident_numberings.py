"""The on-chip solvers on meshes that are not numbered row by row: reverse
Cuthill-McKee, which has no row length, so that rows go to blocks in strips
whose halo is the bandwidth on either side.  Where that fits a block's shared
memory the solve is on chip (after three iterations only the order of the sums
differs, 1e-12), else it is the other engine's, to the bit."""
import numpy as np
import pytest
import scipy.sparse as sp
from scipy.sparse.csgraph import reverse_cuthill_mckee

from fortranfvcell_amd import problems as P

pytestmark = pytest.mark.gpu


def _rcm(s):
    inner = s.nbr >= 0
    rows = np.repeat(np.arange(s.neq), s.w)[inner.ravel()]
    g = sp.csr_matrix((np.ones(rows.size), (rows, s.nbr[inner])), shape=(s.neq, s.neq))
    p = reverse_cuthill_mckee(g, symmetric_mode=True).astype(np.int64)
    q = np.empty(s.neq, np.int64)
    q[p] = np.arange(s.neq)
    return P.System(s.neq, s.w, s.ad[p], s.off[p], np.where(s.nbr[p] >= 0, q[np.maximum(s.nbr[p], 0)], -1), s.b[p])


# bandwidths of about the shorter side; shared memory holds a halo of 2 x 433 rows
# (BiCGSTAB) or 2 x 884 (PCG) beside eight rows a thread, 2 x 984 or more beside fewer
@pytest.mark.parametrize("nx,ny,method,on_chip", [
    (60, 50, "bicgstab", True), (211, 97, "pcg", True), (230, 231, "gmres", True), (500, 500, "bicgstab", True),
    (500, 500, "pcg", True), (640, 620, "mixed", True), (800, 800, "bicgstab", False), (800, 800, "pcg", True)])
def test_rcm(fvc, nx, ny, method, on_chip):
    m = P.quad_mesh(nx, ny, jitter=0.1, seed=nx)
    s = P.pressure_system(m, k=P.lognormal_k(3, m.neq), pin="penalty") if method in ("pcg", "mixed") else \
        P.advdiff_system(m, dt=0.005, under_relax=0.8)
    f = P.to_ell(_rcm(s))
    code = dict(pcg=fvc.PCG, mixed=fvc.PCG, bicgstab=fvc.BICGSTAB, gmres=fvc.GMRES)[method]
    kw = dict(tol=1e-10, x0_rule=fvc.X0_ZERO, maxit=1 if method == "gmres" else 3)
    if method == "mixed":
        kw["precision"] = fvc.PREC_MIXED
    elif method == "gmres":
        kw["gmres_k"] = 3
    else:
        kw["stop_rule"] = fvc.STOP_RELRES
    print(f"rcm {nx}x{ny} {method}", flush=True)
    xa, sa = fvc.solve(f, code, **kw)
    xk, sk = fvc.solve(f, code, engine=fvc.ENGINE_KERNELS, **kw)
    assert (sa["status"], sa["iterations"]) == (sk["status"], sk["iterations"])
    assert sa["engine"] == (fvc.ENGINE_PERSISTENT if on_chip else fvc.ENGINE_KERNELS)
    if on_chip:
        assert np.linalg.norm(xa - xk) <= (1e-6 if method == "mixed" else 1e-12) * np.linalg.norm(xk)
    else:
        assert np.array_equal(xa, xk)
