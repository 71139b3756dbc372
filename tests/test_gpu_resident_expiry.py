"""What follows when a wait of an on-chip solve expires (fvc_resident.h): the
launch ends, and the other engines solve the system from what the caller gave.
The expiry is forced by the host, which has every wait from a given exchange on
end after one look (fvc_test_expire); every block still leaves by itself."""
import os
import subprocess
import sys

import numpy as np
import pytest

from fortranfvcell_amd import _lib, problems as P

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _expire(exchange):
    _lib.check(_lib.load().fvc_test_expire(exchange))


@pytest.fixture(scope="module")
def uneven():
    """160 systems of several blocks and 400 of one: on 256 CUs nearly every
    block runs systems of one block after those of its teams."""
    sides = [66 + i % 9 for i in range(160)] + [14 + i % 11 for i in range(400)]
    made = {n: P.pressure_system(P.quad_mesh(n), k=P.lognormal_k(n, n * n), seed=n, pin="penalty") for n in set(sides)}
    return [made[n] for n in sides]


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
def test_batch_leaves_whole(fvc, uneven, precision):
    """A block leaves a batch with all of its waves, also where a system that
    it holds alone would be next; solved to the library's bars all the same."""
    batch = fvc.concat_ell([P.to_ell(s) for s in uneven])
    ro = batch["row_offsets"]
    kw = dict(tol=1e-10, stop_rule=fvc.STOP_RELRES, precision=precision)
    xs, ss = fvc.solve_batch(batch, block_size=512, **kw)
    mats = {s.neq: P.scipy_csr(s) for s in uneven}
    for exchange in (1, 2, 3, 17, 100):
        print(f"batch expires from exchange {exchange} on, precision {precision}", flush=True)
        _expire(exchange)
        x, sts = fvc.solve_batch(batch, **kw)
        for i, s in enumerate(uneven):
            xi, yi = x[ro[i]:ro[i + 1]], xs[ro[i]:ro[i + 1]]
            assert sts[i]["status"] == ss[i]["status"] == 0, (i, sts[i])
            assert np.linalg.norm(s.b - mats[s.neq] @ xi) <= 1.01e-10 * np.linalg.norm(s.b), i
            assert np.linalg.norm(xi - yi) <= 1e-8 * np.linalg.norm(yi), i


@pytest.mark.parametrize("code", [1, 2], ids=["pcg", "bicgstab"])
@pytest.mark.parametrize("nx,ny", [(70, 61), (231, 230), (499, 498)])
def test_solve_restarts_from_x0(fvc, nx, ny, code):
    """The other engine starts from the caller's x0 also where some blocks had
    written their x already (a wait of the last exchange): the same bits as that
    engine alone.  Where every word was there at the first look the solve ends on
    chip: the order of the sums only, over three iterations (1e-12)."""
    m = P.quad_mesh(nx, ny, jitter=0.1, seed=nx)
    s = P.pressure_system(m, k=P.lognormal_k(3, m.neq), pin="penalty") if code == 1 else \
        P.advdiff_system(m, dt=0.005, under_relax=0.8)
    f = P.to_ell(s)
    x0 = np.random.default_rng(nx).normal(size=m.neq)
    kw = dict(x0=x0, tol=1e-10, stop_rule=fvc.STOP_RELRES, x0_rule=fvc.X0_GIVEN, maxit=3)
    xk, sk = fvc.solve(f, code, engine=fvc.ENGINE_KERNELS, **kw)
    fell = 0
    for exchange in range(1, 12):
        print(f"{nx}x{ny} code={code} expires from exchange {exchange} on", flush=True)
        for _ in range(4):
            _expire(exchange)
            xa, sa = fvc.solve(f, code, **kw)
            assert (sa["status"], sa["iterations"]) == (sk["status"], sk["iterations"]) == (1, 3)
            if sa["engine"] == fvc.ENGINE_KERNELS:
                fell += 1
                assert np.array_equal(xa, xk)
            else:
                assert np.linalg.norm(xa - xk) <= 1e-12 * np.linalg.norm(xk)
    assert fell > 0


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
def test_batch_restarts_from_x0(fvc, uneven, precision):
    """As above: an expired wait sends every system of the batch to the other
    kernels, those whose x was written too.  After three iterations the order of
    the sums only (FP64 1e-12; FP32 vectors may round the other way, 1e-6)."""
    batch = fvc.concat_ell([P.to_ell(s) for s in uneven])
    ro = batch["row_offsets"]
    x0 = np.random.default_rng(1).normal(size=int(ro[-1]))
    x0[batch["ad"] > 1e50] = 0.0   # the pinned rows hold it
    kw = dict(x0=x0, tol=1e-10, stop_rule=fvc.STOP_RELRES, x0_rule=fvc.X0_GIVEN, precision=precision, maxit=3)
    xs, ss = fvc.solve_batch(batch, block_size=512, **kw)
    for exchange in range(1, 10):
        print(f"batch expires from exchange {exchange} on, precision {precision}", flush=True)
        _expire(exchange)
        x, sts = fvc.solve_batch(batch, **kw)
        for i in range(len(uneven)):
            xi, yi = x[ro[i]:ro[i + 1]], xs[ro[i]:ro[i + 1]]
            assert (sts[i]["status"], sts[i]["iterations"]) == (ss[i]["status"], ss[i]["iterations"]) == (1, 3), i
            assert np.linalg.norm(xi - yi) <= (1e-12 if precision == 0 else 1e-6) * np.linalg.norm(yi), i



# (a process of its own: torch's HIP runtime has to be loaded first)
BESIDE = r"""
import sys, time
import torch
import numpy as np
import fortranfvcell_amd as F
from fortranfvcell_amd import problems as P
code = int(sys.argv[1])
F.init(0)
s = P.config_advdiff(1024)
ds = F.DeviceSystem(P.to_ell(s))
kw = dict(tol=1e-10, stop_rule=F.STOP_RELRES, x0_rule=F.X0_ZERO)
assert ds.solve(code, **kw)["engine"] == F.ENGINE_PERSISTENT
torch.cuda._sleep(1000)
torch.cuda.synchronize()
t = time.perf_counter()
torch.cuda._sleep(10_000_000)
torch.cuda.synchronize()
cycles = int(0.8 * 1e7 / (time.perf_counter() - t))
side = torch.cuda.Stream()
with torch.cuda.stream(side):
    torch.cuda._sleep(cycles)
time.sleep(0.01)
t = time.perf_counter()
st = ds.solve(code, **kw)
t = time.perf_counter() - t
asleep = not side.query()
side.synchronize()
r = np.linalg.norm(s.b - P.scipy_csr(s) @ ds.x.get()) / np.linalg.norm(s.b)
print("result", t, int(asleep), st["status"], st["engine"], r)
"""


@pytest.mark.parametrize("code", [2, 3], ids=["bicgstab", "gmres"])
def test_solve_beside_a_long_kernel(code):
    """A wave of another stream, asleep for 0.8 s, keeps one of the 256 blocks off
    the chip (blocks of eight rows a thread take all of a CU's registers): the
    solve does not wait for it but goes to an engine that needs no CU to itself,
    which takes 3 ms (BiCGSTAB) and 25 ms (GMRES) alone."""
    r = subprocess.run([sys.executable, "-c", BESIDE, str(code)], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    t, asleep, status, engine, relres = (float(v) for v in r.stdout.split("result")[1].split())
    print(f"code {code}: {t * 1e3:.1f} ms, engine {engine:.0f}, other stream still busy {asleep:.0f}", flush=True)
    assert asleep == 1 and t < 0.2 and status == 0 and relres <= 1.01e-10
