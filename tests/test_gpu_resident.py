"""PCG and BiCGSTAB held on chip (fvc_resident.h), which AUTO takes where the
system fits: against the engine that runs one kernel per phase, at the edges
of what a block, a launch and a tile hold, for every layout that takes this
path, both starting points and a capped iteration count.

Bars: after three iterations only the order of the sums differs, so x agrees
to 1e-12 (a few hundred roundings of sums of up to 300,000 terms); solved to a
true residual of 1e-10, ||x - x'|| <= 1e-8 ||x'||, the library's bar for
solutions."""
import numpy as np
import pytest

from fortranfvcell_amd import problems as P

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def _mesh(kind, nx, ny):
    return P.quad_mesh(nx, ny, jitter=0.1, seed=nx) if kind == "quad" else P.tri_mesh(nx, jitter=0.1, seed=nx)


# one row; one thread's, two's, four's rows of one block and just beyond (2,048
# rows); up to 64 blocks and just beyond; rows per thread 2 -> 4 (249k rows) and
# 4 -> 8; long, thin meshes (strips, wide and narrow tiles)
SHAPES = [("quad", 1, 1), ("quad", 3, 2), ("quad", 32, 16), ("quad", 27, 19), ("quad", 32, 32), ("quad", 64, 32),
          ("quad", 41, 50), ("tri", 37, 0), ("quad", 13, 2041), ("quad", 2041, 13), ("quad", 163, 163),
          ("quad", 231, 230), ("tri", 170, 0), ("quad", 499, 498), ("quad", 499, 501), ("tri", 500, 0)]


@pytest.mark.parametrize("kind,nx,ny", SHAPES)
@pytest.mark.parametrize("code", [1, 2], ids=["pcg", "bicgstab"])
def test_resident_matches_kernels(fvc, kind, nx, ny, code):
    m = _mesh(kind, nx, ny)
    s = P.pressure_system(m, k=P.lognormal_k(3, m.neq), pin="penalty") if code == 1 else \
        P.advdiff_system(m, dt=0.005, under_relax=0.8) if m.neq > 1 else P.pressure_system(m, pin="identity")
    if code == 1 and m.neq == 1:
        s = P.pressure_system(m, pin="identity")
        s.b[:] = 2.0
    x0 = np.random.default_rng(nx).normal(size=m.neq)
    for lay in (P.to_ell, P.to_csrd):
        f = lay(s)
        for opt in (dict(x0_rule=fvc.X0_ZERO, maxit=3), dict(x0_rule=fvc.X0_GIVEN, maxit=3),
                    dict(x0_rule=fvc.X0_ZERO), dict(x0_rule=fvc.X0_GIVEN)):
            if "maxit" not in opt and code == 1 and m.neq > 60000:
                continue
            print(f"resident {kind} {nx}x{ny} neq={m.neq} code={code} {lay.__name__} {opt}", flush=True)
            kw = dict(tol=1e-10, stop_rule=fvc.STOP_RELRES, **opt)
            xa, sa = fvc.solve(f, code, x0=x0, **kw)
            xk, sk = fvc.solve(f, code, x0=x0, engine=fvc.ENGINE_KERNELS, **kw)
            assert sa["status"] == sk["status"] and sk["engine"] == fvc.ENGINE_KERNELS
            # a breakdown (BiCGSTAB on one row) is left to the other engine
            assert sa["engine"] == (fvc.ENGINE_PERSISTENT if sa["status"] <= 1 else fvc.ENGINE_KERNELS)
            capped = "maxit" in opt
            assert _rel(xa, xk) <= (1e-12 if capped else 1e-8), (opt, sa, sk)
            if capped:
                assert sa["iterations"] == sk["iterations"]
                assert abs(sa["energy"] - sk["energy"]) <= 1e-10 * abs(sk["energy"])
            elif sa["status"] == 0:
                assert sa["true_relres"] <= 1e-10


@pytest.mark.parametrize("n", [(24, 23), (113, 90), (400, 380)], ids=["one_block", "few_blocks", "many_blocks"])
def test_resident_repeats_bit_for_bit(fvc, n):
    s = P.advdiff_system(_mesh("quad", *n), dt=0.005, under_relax=0.8)
    ds = fvc.DeviceSystem(P.to_ell(s))
    xs = []
    for _ in range(3):
        ds.solve(fvc.BICGSTAB, tol=1e-11, stop_rule=fvc.STOP_RELRES, x0_rule=fvc.X0_ZERO)
        xs.append(ds.x.get())
    assert np.array_equal(xs[0], xs[1]) and np.array_equal(xs[0], xs[2])


def test_resident_declines_what_does_not_fit(fvc):
    """Columns far apart (a random numbering), and rows of more than four
    off-diagonals: solved one kernel per phase, the same answer."""
    s = P.config_pressure_lognormal(100)
    p = np.random.default_rng(5).permutation(s.neq)
    q = np.empty(s.neq, np.int64)
    q[p] = np.arange(s.neq)
    nbr = np.where(s.nbr[p] >= 0, q[np.maximum(s.nbr[p], 0)], -1)
    renum = P.System(s.neq, s.w, s.ad[p], s.off[p], nbr, s.b[p])
    x, st = fvc.solve(P.to_ell(renum), fvc.PCG, tol=1e-10, stop_rule=fvc.STOP_RELRES, x0_rule=fvc.X0_ZERO)
    assert st["engine"] == fvc.ENGINE_KERNELS and st["status"] == 0 and st["true_relres"] <= 1e-10
    # a 9-point operator in CSRD: eight off-diagonals a row, in one block and in several
    import scipy.sparse as sp
    for n in (16, 70):
        t = sp.diags([-1.0, 2.5, -1.0], [-1, 0, 1], shape=(n, n))
        A = sp.kron(t, t).tocsr()
        A.sort_indices()
        d = A.diagonal()
        off = (A - sp.diags(d)).tocsr()
        off.eliminate_zeros()
        off.sort_indices()
        b = np.random.default_rng(n).normal(size=n * n)
        f = dict(matriz=1, neq=n * n, nad=off.nnz, iax=(off.indptr + 1).astype(np.int32),
                 ja=(off.indices + 1).astype(np.int32), ad=d, al=off.data.copy(), au=None, b=b, sym=False)
        x, st = fvc.solve(f, fvc.PCG, tol=1e-10, stop_rule=fvc.STOP_RELRES, x0_rule=fvc.X0_ZERO, maxit=20000)
        assert st["engine"] == fvc.ENGINE_KERNELS and st["status"] == 0
        assert np.linalg.norm(b - A @ x) <= 1.01e-10 * np.linalg.norm(b)


def test_resident_reports_breakdown_and_nonfinite(fvc):
    """Left to one kernel per phase, whose status the caller gets, in one block
    and in several; x0 is what that engine starts from."""
    for n in (16, 70):
        s = P.config_advdiff(n, peclet_max=10.0)
        f = P.to_ell(s)
        for b in (np.zeros(s.neq), np.where(np.arange(s.neq) == 3, np.nan, 1.0)):
            for code in (1, 2):
                for stop in (fvc.STOP_RELRES, fvc.STOP_REFERENCE):
                    kw = dict(b=b, tol=1e-10, stop_rule=stop, x0_rule=fvc.X0_ZERO, maxit=50)
                    _, sa = fvc.solve(f, code, **kw)
                    _, sk = fvc.solve(f, code, engine=fvc.ENGINE_KERNELS, **kw)
                    assert (sa["status"], sa["iterations"]) == (sk["status"], sk["iterations"]), (n, code, stop)
                    if sa["status"] > 1:
                        assert sa["engine"] == fvc.ENGINE_KERNELS


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("given", [False, True], ids=["x0_zero", "x0_given"])
def test_resident_batch_beside_systems_that_do_not_fit(fvc, given, precision):
    """One launch takes the systems that fit, whatever their team (one block,
    a few, many), and the streaming kernels the others (a random numbering)."""
    sides = [1, 3, 8, 22, 23, 33, 46, 64, 91, 130, 201]
    systems = [P.pressure_system(P.quad_mesh(n), k=P.lognormal_k(n, n * n), seed=n, pin="penalty" if n > 1 else "identity")
               for n in sides]
    s = P.config_pressure_lognormal(60)
    p = np.random.default_rng(5).permutation(s.neq)
    q = np.empty(s.neq, np.int64)
    q[p] = np.arange(s.neq)
    systems.insert(4, P.System(s.neq, s.w, s.ad[p], s.off[p], np.where(s.nbr[p] >= 0, q[np.maximum(s.nbr[p], 0)], -1), s.b[p]))
    systems[0].b[:] = 3.0
    for lay, cat in ((P.to_ell, fvc.concat_ell), (P.to_csrd, fvc.concat_csrd)):
        batch = cat([lay(t) for t in systems])
        n = int(batch["row_offsets"][-1])
        x0 = np.random.default_rng(1).normal(size=n) if given else None
        if given:
            # where the 1e60 pin holds it: off it, the pinned row's residual is 1e60
            # and no recursive residual of the solve knows what rounding left of it
            x0[batch["ad"] > 1e50] = 0.0
        kw = dict(tol=1e-10, stop_rule=fvc.STOP_RELRES, x0_rule=fvc.X0_GIVEN if given else fvc.X0_ZERO,
                  precision=precision)
        print(f"resident batch of {len(systems)} systems {lay.__name__} given={given}", flush=True)
        x, sts = fvc.solve_batch(batch, x0=x0, **kw)
        xs, ss = fvc.solve_batch(batch, x0=x0, block_size=256, **kw)
        ro = batch["row_offsets"]
        for i, t in enumerate(systems):
            xi, yi = x[ro[i]:ro[i + 1]], xs[ro[i]:ro[i + 1]]
            assert sts[i]["status"] == ss[i]["status"], (i, sts[i], ss[i])
            if sts[i]["status"] != 0:   # (the FP32 recursion of 9 rows overflows, in either engine)
                assert precision == 1 and t.neq <= 9
                continue
            assert np.linalg.norm(t.b - P.scipy_csr(t) @ xi) <= 1.01e-10 * np.linalg.norm(t.b), i
            assert np.linalg.norm(xi - yi) <= 1e-8 * np.linalg.norm(yi), i


def test_resident_batch_maxit(fvc):
    systems = [P.pressure_system(P.quad_mesh(n), seed=n) for n in (10, 40, 90)]
    batch = fvc.concat_ell([P.to_ell(s) for s in systems])
    x, sts = fvc.solve_batch(batch, tol=1e-10, maxit=5, stop_rule=fvc.STOP_RELRES)
    xs, ss = fvc.solve_batch(batch, tol=1e-10, maxit=5, stop_rule=fvc.STOP_RELRES, block_size=256)
    assert [(s["status"], s["iterations"]) for s in sts] == [(s["status"], s["iterations"]) for s in ss] == [(1, 5)] * 3
    assert np.linalg.norm(x - xs) <= 1e-12 * np.linalg.norm(xs)


@pytest.mark.parametrize("kind,nx,ny", SHAPES[1:])
def test_resident_mixed_matches_kernels(fvc, kind, nx, ny):
    """Mixed precision on chip: the same FP32 rows and vectors, so that after
    three iterations only the FP64 sums' order differs (a step length moved by
    1e-15 may round an FP32 vector the other way: 1e-6); solved, the true FP64
    residual and the library's bar for solutions.  A start vector is kept for
    a solve that is declined (here: none), and maxit counts FP32 iterations."""
    m = _mesh(kind, nx, ny)
    s = P.pressure_system(m, k=P.lognormal_k(3, m.neq))
    x0 = np.random.default_rng(nx).normal(size=m.neq)
    x0[0] = 0.0   # the pinned cell
    for lay in (P.to_ell, P.to_csrd):
        f = lay(s)
        for opt in (dict(x0_rule=fvc.X0_ZERO, maxit=3), dict(x0_rule=fvc.X0_GIVEN, maxit=3),
                    dict(x0_rule=fvc.X0_ZERO), dict(x0_rule=fvc.X0_GIVEN)):
            if "maxit" not in opt and m.neq > 60000:
                continue
            print(f"resident mixed {kind} {nx}x{ny} neq={m.neq} {lay.__name__} {opt}", flush=True)
            kw = dict(tol=1e-10, precision=fvc.PREC_MIXED, **opt)
            xa, sa = fvc.solve(f, fvc.PCG, x0=x0, **kw)
            xk, sk = fvc.solve(f, fvc.PCG, x0=x0, engine=fvc.ENGINE_KERNELS, **kw)
            assert sa["status"] == sk["status"] and sa["flags"] & fvc.FLAG_COL16 == sk["flags"] & fvc.FLAG_COL16
            if sa["engine"] == fvc.ENGINE_KERNELS:
                # the FP32 recursion of a few rows overflows past its solution, or does
                # not, by a rounding: declined, so exactly the other engine's outcome
                assert m.neq <= 9 and np.array_equal(xa, xk, equal_nan=True)
                continue
            assert sa["status"] <= 1
            capped = "maxit" in opt
            assert _rel(xa, xk) <= (1e-6 if capped else 1e-8), (opt, sa, sk)
            if capped:
                assert sa["iterations"] == sk["iterations"] == 3
            elif sa["status"] == 0:   # (the 2,738 triangles reach maxit in every engine)
                assert sa["true_relres"] <= 1e-10


def test_resident_mixed_declines(fvc):
    """A random numbering, warm-started: x0 reaches the other engine as given."""
    s = P.config_pressure_lognormal(70)
    p = np.random.default_rng(5).permutation(s.neq)
    q = np.empty(s.neq, np.int64)
    q[p] = np.arange(s.neq)
    renum = P.System(s.neq, s.w, s.ad[p], s.off[p], np.where(s.nbr[p] >= 0, q[np.maximum(s.nbr[p], 0)], -1), s.b[p])
    f = P.to_ell(renum)
    x, st = fvc.solve(f, fvc.PCG, tol=1e-10, precision=fvc.PREC_MIXED, x0_rule=fvc.X0_ZERO)
    assert st["engine"] == fvc.ENGINE_KERNELS and st["status"] == 0
    x2, st2 = fvc.solve(f, fvc.PCG, x0=x, tol=1e-10, precision=fvc.PREC_MIXED, x0_rule=fvc.X0_GIVEN)
    assert st2["iterations"] == 0 and np.array_equal(x2, x)


@pytest.mark.parametrize("kind,nx,ny", SHAPES[2:])
@pytest.mark.parametrize("k", [1, 2, 3, 15, 32])
def test_resident_gmres_matches_kernels(fvc, kind, nx, ny, k):
    """Modified Gram-Schmidt on chip against one kernel per phase: the same
    steps, and after one cycle x to 1e-11 (sums in another order, of
    vectors of norm one, over k projections); the restart lengths around the
    prefetch of columns, and the longest that the chip takes."""
    m = _mesh(kind, nx, ny)
    s = P.advdiff_system(m, dt=0.005, under_relax=0.8)
    for lay in (P.to_ell, P.to_csrd):
        f = lay(s)
        for opt in (dict(maxit=1, stop_rule=fvc.STOP_REFERENCE), dict(maxit=400, stop_rule=fvc.STOP_RELRES)):
            if opt["maxit"] > 1 and (k < 15 or m.neq > 60000):
                continue
            print(f"resident gmres({k}) {kind} {nx}x{ny} neq={m.neq} {lay.__name__} {opt}", flush=True)
            kw = dict(tol=1e-10, gmres_k=k, **opt)
            xa, sa = fvc.solve(f, fvc.GMRES, **kw)
            xk, sk = fvc.solve(f, fvc.GMRES, engine=fvc.ENGINE_KERNELS, **kw)
            assert (sa["status"], sa["iterations"], sa["inner_iterations"]) == \
                (sk["status"], sk["iterations"], sk["inner_iterations"]), (sa, sk)
            assert _rel(xa, xk) <= (1e-11 if opt["maxit"] == 1 else 1e-8)
            assert abs(sa["energy"] - sk["energy"]) <= 1e-8 * abs(sk["energy"])
            if opt["maxit"] > 1:
                assert sa["true_relres"] <= 1e-10


def test_resident_gmres_exact_start(fvc):
    """A zero right-hand side: the exact solution at once, in either engine."""
    for n in (20, 70):
        f = P.to_ell(P.config_advdiff(n, peclet_max=10.0))
        x, st = fvc.solve(f, fvc.GMRES, b=np.zeros(n * n), tol=1e-10, gmres_k=10)
        xk, sk = fvc.solve(f, fvc.GMRES, b=np.zeros(n * n), tol=1e-10, gmres_k=10, engine=fvc.ENGINE_KERNELS)
        assert (st["status"], st["iterations"]) == (sk["status"], sk["iterations"]) and not x.any() and not xk.any()


@pytest.mark.parametrize("kind,nx,ny", [("quad", 208, 128), ("quad", 213, 125), ("quad", 253, 257), ("quad", 256, 256),
                                        ("quad", 64, 1024), ("quad", 6001, 10), ("quad", 257, 256), ("tri", 181, 0),
                                        ("quad", 512, 256), ("quad", 361, 363), ("quad", 171, 767)])
def test_resident_at_the_edges_of_64_blocks(fvc, kind, nx, ny):
    """Plans of at most 64 blocks are preferred: one, two and (PCG) four rows
    a thread at the last rows that 52 and 64 blocks hold and just beyond, in
    tiles and in strips.  After two iterations only the order of the sums differs (1e-12, as above)."""
    m = _mesh(kind, nx, ny)
    sp = P.pressure_system(m, k=P.lognormal_k(3, m.neq), pin="penalty")
    sm = P.advdiff_system(m, dt=0.005, under_relax=0.8)
    for code, s in ((fvc.PCG, sp), (fvc.BICGSTAB, sm)):
        f = P.to_ell(s)
        print(f"64 blocks {kind} {nx}x{ny} neq={m.neq} code={code}", flush=True)
        kw = dict(tol=1e-10, stop_rule=fvc.STOP_RELRES, x0_rule=fvc.X0_ZERO, maxit=2)
        xa, sa = fvc.solve(f, code, **kw)
        xk, sk = fvc.solve(f, code, engine=fvc.ENGINE_KERNELS, **kw)
        assert sa["engine"] == fvc.ENGINE_PERSISTENT and sa["iterations"] == sk["iterations"] == 2
        assert _rel(xa, xk) <= 1e-12


@pytest.mark.parametrize("n", [108, 301, 392])
def test_resident_finds_the_row_length(fvc, n):
    """Triangles split from quads, 2 n cells to a row, at sizes where rows
    spread evenly over the system miss every place where 2 n - 1 wraps: tiles
    of that length would hold columns outside their window."""
    m = _mesh("tri", n, 0)
    s = P.advdiff_system(m, dt=0.005, under_relax=0.8)
    kw = dict(tol=1e-10, stop_rule=fvc.STOP_RELRES, x0_rule=fvc.X0_ZERO, maxit=2)
    for lay in (P.to_ell, P.to_csrd):
        f = lay(s)
        for code in (fvc.PCG, fvc.BICGSTAB):
            print(f"row length tri {n} {lay.__name__} code={code}", flush=True)
            xa, sa = fvc.solve(f, code, **kw)
            xk, sk = fvc.solve(f, code, engine=fvc.ENGINE_KERNELS, **kw)
            assert sa["engine"] == fvc.ENGINE_PERSISTENT and sa["iterations"] == sk["iterations"] == 2
            assert _rel(xa, xk) <= 1e-12
