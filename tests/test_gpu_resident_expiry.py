"""What follows when a wait of an on-chip solve expires (fvc_resident.h): the
launch ends, and the other engines solve the system from what the caller gave.
The expiry is forced by the host, which has every wait from a given exchange on
end after one look (fvc_test_expire); every block still leaves by itself."""
import numpy as np
import pytest

from fortranfvcell_amd import _lib, problems as P

pytestmark = pytest.mark.gpu


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
