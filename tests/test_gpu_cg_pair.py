"""Two right-hand sides in the same CG launches against two separate solves.

SPLR's low-rank solve (src/sinkhorn_linsolve.cpp:160-225) solves the Newton
system for two right-hand sides.  The GPU runs both CGs in the same kernel
launches (grid row 0 and 1), each with its own vectors, scalars and stop
test, so each must return exactly what a CG of its own returns: the same
solution bit for bit, the same iteration count and the same residual, also
when one side stops long before the other, hits the cap, has a zero
right-hand side or is already converged at the start.  Matrix-free Hessians
run the two solves one after the other.
"""
import numpy as np
import pytest

from conftest import cloud_problem

pytestmark = pytest.mark.gpu


def near_optimum(P):
    from regot import _lib
    return P.solve(_lib.SOLVER_BCD, tol=1e-5, max_iter=5000, compute_plan=False).dual


def same(single, pair, k):
    x, it, err = single
    (x0, x1), its, errs = pair
    xs = (x0, x1)[k]
    assert its[k] == it
    assert errs[k] == err
    assert np.array_equal(xs, x)


@pytest.mark.parametrize("bulk", ["fp32", "fp64"])
def test_cg_pair_matches_single_solves(gpu_lib, bulk):
    n, m, reg = 700, 900, 0.02
    M, a, b = cloud_problem(n, m, d=8, seed=81)
    if bulk == "fp32":
        M = M.astype(np.float32)
    rng = np.random.default_rng(8)
    N = n + m - 1
    with gpu_lib.Problem(M, a, b, reg) as P:
        P.set_hess_storage(0)
        gamma = near_optimum(P)
        P.sparsified_hess_with_density(gamma, 0.02)
        h2max = P.hess_export()["h2"].max()
        # (shift scale, tol, cap, rhs1 kind): both long; different lengths
        # (the second right-hand side nearly constant); a cap that ends both;
        # a zero right-hand side; both converged at the start (tol > 1)
        cases = [(1e-4, 1e-12, 5000, "rand"), (1e-3, 1e-10, 5000, "smooth"),
                 (1e-5, 1e-12, 37, "rand"), (1e-3, 1e-10, 5000, "zero"),
                 (1e-3, 2.0, 5000, "rand")]
        for q, (sc, tol, cap, kind) in enumerate(cases):
            shift = sc * h2max
            r0 = rng.standard_normal(N)
            if kind == "rand":
                r1 = rng.standard_normal(N)
            elif kind == "smooth":
                r1 = np.ones(N) + 1e-3 * rng.standard_normal(N)
            else:
                r1 = np.zeros(N)
            print(f"cg pair {bulk} case {q}: {kind}", flush=True)
            s0 = P.hess_cg(r0, shift, tol=tol, max_iter=cap)
            s1 = P.hess_cg(r1, shift, tol=tol, max_iter=cap)
            pr = P.hess_cg2(r0, r1, shift, tol=tol, max_iter=cap)
            print(f"  iterations {s0[1]} / {s1[1]}", flush=True)
            same(s0, pr, 0)
            same(s1, pr, 1)
            if q == 2:
                assert s0[1] == cap and s1[1] == cap
            if kind == "zero":
                assert s1[1] == 0 and np.all(pr[0][1] == 0.0)
            if tol > 1:
                assert s0[1] == 0 and s1[1] == 0
            elif kind != "zero":
                assert s0[1] > 16 and s1[1] > 16   # past the first batch


def test_cg_pair_matrix_free_runs_two_solves(gpu_lib):
    n, m, reg = 400, 600, 0.05
    M, a, b = cloud_problem(n, m, seed=82)
    M32 = M.astype(np.float32)
    rng = np.random.default_rng(9)
    N = n + m - 1
    with gpu_lib.Problem(M32, a, b, reg) as P:
        P.set_hess_storage(1)
        gamma = near_optimum(P)
        P.sparsified_hess_with_density(gamma, 1.0)
        r0, r1 = rng.standard_normal(N), rng.standard_normal(N)
        shift = 1e-3
        s0 = P.hess_cg(r0, shift, tol=1e-10, max_iter=5000)
        s1 = P.hess_cg(r1, shift, tol=1e-10, max_iter=5000)
        pr = P.hess_cg2(r0, r1, shift, tol=1e-10, max_iter=5000)
    same(s0, pr, 0)
    same(s1, pr, 1)


@pytest.mark.parametrize("bulk,n,m,density", [("fp32", 3001, 3503, 0.1), ("fp64", 3001, 3503, 0.1),
                                              ("fp32", 16387, 2050, 0.12),
                                              ("fp32", 18431, 11000, 0.005)])
def test_cg_products_with_vector_in_lds(gpu_lib, bulk, n, m, density):
    """Sets of more than 1 M stored entries, whose products keep the gathered
    vector in LDS: odd sizes, a last workgroup with few rows, one and two
    right-hand sides, against the residual formed from the exported entries."""
    import scipy.sparse as sp
    reg = 0.02
    M, a, b = cloud_problem(n, m, d=8, seed=82)
    if bulk == "fp32":
        M = M.astype(np.float32)
    rng = np.random.default_rng(9)
    N, tol = n + m - 1, 1e-10
    with gpu_lib.Problem(M, a, b, reg) as P:
        P.set_hess_storage(0)
        P.sparsified_hess_with_density(near_optimum(P), density)
        H = P.hess_export()
        assert len(H["rval"]) > 1000000
        S = sp.csr_matrix((H["rval"], H["colind"], H["rowptr"]), shape=(n, m - 1))
        shift = 1e-3 * H["h2"].max()
        r0, r1 = rng.standard_normal(N), rng.standard_normal(N)
        s0 = P.hess_cg(r0, shift, tol=tol, max_iter=2000)
        s1 = P.hess_cg(r1, shift, tol=tol, max_iter=2000)
        pr = P.hess_cg2(r0, r1, shift, tol=tol, max_iter=2000)
        same(s0, pr, 0)
        same(s1, pr, 1)
        for r, (x, it, err) in ((r0, s0), (r1, s1)):
            assert 0 < it < 2000 and err <= tol
            # the residual of the eliminated system, relative to its right-hand side
            d1 = H["h1"] + shift
            rhs = r[n:] - S.T @ (r[:n] / d1)
            res = rhs - ((H["h2"] + shift) * x[n:] - S.T @ ((S @ x[n:]) / d1))
            # the recurrence's residual drifts from the true one by rounding:
            # it steps of 2^-52 times the size of Delta x (|Delta| <= 2 max h2)
            drift = it * 2.0 ** -50 * 2.0 * H["h2"].max() * np.linalg.norm(x[n:])
            assert np.linalg.norm(res) <= tol * np.linalg.norm(rhs) + drift
            top = (r[:n] - S @ x[n:]) / d1
            assert np.allclose(x[:n], top, rtol=1e-12, atol=1e-12 * np.abs(top).max())


# 64 lanes per row in both products (up to 8192 rows, or many entries a row), in the
# columns alone (18431 x 11000, 0.5%) or the rows' (2050 x 18433), sets below the usual line, a row and a column
# more than a multiple of 4 per workgroup, the longest vector
@pytest.mark.parametrize("bulk,n,m,density,both", [
    ("fp32", 3001, 3503, 0.1, True), ("fp64", 3001, 3503, 0.1, True),
    ("fp32", 1025, 258, 0.02, True), ("fp64", 700, 901, 0.03, True),
    ("fp32", 16387, 2050, 0.12, True), ("fp64", 2050, 18433, 0.02, False),
    ("fp32", 18431, 11000, 0.005, False), ("fp32", 5, 3, 1.0, True)])
def test_cg_products_in_lds_give_the_same_bits(gpu_lib, bulk, n, m, density, both):
    reg = 0.02
    M, a, b = cloud_problem(n, m, d=8, seed=83)
    if bulk == "fp32":
        M = M.astype(np.float32)
    rng = np.random.default_rng(10)
    N = n + m - 1
    print("cg lds bits %dx%d %s" % (n, m, bulk), flush=True)
    with gpu_lib.Problem(M, a, b, reg) as P:
        P.set_hess_storage(0)
        P.sparsified_hess_with_density(near_optimum(P), density)
        shift = 1e-3 * P.hess_export()["h2"].max()
        r0, r1 = rng.standard_normal(N), rng.standard_normal(N)
        # a cap inside a batch of iterations, both ends of a solve, a pair
        runs = [lambda: P.hess_cg(r0, shift, tol=1e-10, max_iter=2000),
                lambda: P.hess_cg(r1, shift, tol=1e-10, max_iter=5),
                lambda: P.hess_cg2(r0, r1, shift, tol=1e-10, max_iter=2000)]
        P.cg_lds(1 << 62)
        c0 = P.cg_lds()
        old = [f() for f in runs]
        c1 = P.cg_lds()
        P.cg_lds(0)
        new = [f() for f in runs]
        c2 = P.cg_lds()
    assert c1 == c0
    # both products, or one, of every iteration; what is enqueued past the stop
    # counts too
    its = old[0][1] + old[1][1] + max(old[2][1])
    assert c2 - c1 >= (2 if both else 1) * its > 0
    if not both:
        assert c2 - c1 < 2 * its
    for x, y in zip(old[:2], new[:2]):
        assert np.array_equal(x[0], y[0]) and x[1:] == y[1:]
    assert np.array_equal(old[2][0], new[2][0]) and old[2][1:] == new[2][1:]
