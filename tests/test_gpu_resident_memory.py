"""Device memory of solves that cannot be held on chip: what the engine that
runs them needs, nothing for the on-chip solver's words or its copy of x.  Each
case in a process of its own, since the workspace only grows; the bound is the
vectors of that engine and 4 MiB for its small arrays (under 1 MiB) and the
allocator's granularity (2 MiB).  Reserving the words took 32 bytes a row more,
the copy of x 8."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# bytes a row of the vectors: GMRES(10) FP64 11 columns and x (CSR: and the
# diagonal taken out of the matrix); mixed PCG of width 4 the FP32 and FP64
# scalings, records, FP32 values and int16 columns
CASES = {
    # beyond the chip
    "gmres_beyond": (96, "gmres", "quad", 1100, 1000, {}),
    "mixed_beyond": (68, "mixed", "quad", 1100, 1000, {}),
    # an option that shapes the launch
    "gmres_kernels": (96, "gmres", "quad", 700, 500, dict(engine=1)),
    "gmres_blocks": (96, "gmres", "quad", 700, 500, dict(grid_blocks=128)),
    "mixed_blocks": (68, "mixed", "quad", 900, 800, dict(block_size=256)),
    # a format, and rows, that it does not take
    "gmres_csr": (104, "gmres", "csr", 700, 500, {}),
    "gmres_nine_points": (96, "gmres", "nine", 600, 600, {}),
}

CHILD = r"""
import ctypes, sys
import numpy as np
import scipy.sparse as sp
import fortranfvcell_amd as F
from fortranfvcell_amd import problems as P

method, kind, nx, ny, opt = eval(sys.argv[1])

def system(nx, ny):
    if kind == "nine":
        t = [sp.diags([-1.0, 2.5, -1.0], [-1, 0, 1], shape=(n, n)) for n in (nx, ny)]
        A = sp.kron(t[1], t[0]).tocsr()
        A.sort_indices()
        d = A.diagonal()
        off = (A - sp.diags(d)).tocsr()
        off.eliminate_zeros()
        off.sort_indices()
        return dict(matriz=1, neq=nx * ny, nad=off.nnz, iax=(off.indptr + 1).astype(np.int32),
                    ja=(off.indices + 1).astype(np.int32), ad=d, al=off.data.copy(), au=None, b=np.ones(nx * ny), sym=False)
    s = P.advdiff_system(P.quad_mesh(nx, ny), dt=0.005, under_relax=0.8)
    return P.to_csr(s) if kind == "csr" else P.to_ell(s)

def solve(ds, **o):
    if method == "gmres":
        ds.solve(F.GMRES, gmres_k=10, maxit=1, tol=1e-30, **o)
    else:
        ds.solve(F.PCG, precision=F.PREC_MIXED, maxit=2, tol=1e-30, x0_rule=F.X0_GIVEN, **o)

F.init(0)
with open("/proc/self/maps") as fh:
    hip = ctypes.CDLL(next(w for w in fh.read().split() if "libamdhip64" in w))

def free():
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
    return a.value

small, big = F.DeviceSystem(system(20, 20)), F.DeviceSystem(system(nx, ny))
for e in (0, 1, 2):   # every kernel loaded
    solve(small, engine=e)
before = free()
solve(big, **opt)
print("bytes", before - free(), big.neq)
"""


@pytest.mark.parametrize("name", CASES)
def test_workspace_of_streamed_solves(name):
    per_row, *case = CASES[name]
    print(name, case, flush=True)
    r = subprocess.run([sys.executable, "-c", CHILD, repr(tuple(case))], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    took, neq = (int(v) for v in r.stdout.split("bytes")[1].split())
    print(f"{name}: {took} bytes, {took / neq:.1f} a row", flush=True)
    assert took <= per_row * neq + (4 << 20)
