"""GPU parity of the single-read BCD iteration (one pass over M per iteration).

The FP32 BCD driver runs the single-read form wherever it is eligible
(``bcd_fused``, default 1); ``bcd_fused=0`` keeps the two-pass form.  Checked here against the FP64 oracle (same iteration
semantics, same stop test) and against the two-pass GPU path, on shapes that
cover every column-vector count (m up to 16384, full-width and ragged), the
rows whose range check falls back to an exact row maximum, a warm start, the
eligibility fallback and workgroups holding more rows than threads.
"""
import numpy as np
import pytest

from conftest import cloud_problem
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def rel_err(x, ref):
    return np.max(np.abs(np.asarray(x) - ref)) / max(1.0, np.max(np.abs(ref)))


def fused_expected(r):
    """Single-read passes a solve runs: one per iteration up to the iterate
    where an FP32 solve hands over to its FP64 finish, that one included."""
    pf = r.stats["precise_from"]
    return (pf if pf >= 0 else r.niter) + 1


def solve(gpu_lib, M, a, b, reg, tol, max_iter, fused, x0=None):
    """BCD through a problem handle with kernel profiling on; returns the
    result and the number of single-read passes that ran."""
    kw = {"bcd_fused": fused}
    if x0 is not None:
        kw["x0"] = x0
    with gpu_lib.Problem(M, a, b, reg) as P:
        P.profile(True)
        r = P.solve(0, tol=tol, max_iter=max_iter, compute_plan=False, verify=True, **kw)
        fused_launches = P.profile_stats(2)[0]
    return r, fused_launches


# (n, m, reg): m covers NC = ceil(m / 2048) = 1, 3, 7, 8, full-width and ragged
SHAPES = [(50, 1500, 0.05), (130, 2048, 0.05), (257, 5000, 0.02), (301, 12289, 0.05),
          (64, 16384, 0.05), (90, 14500, 0.05)]


@pytest.mark.parametrize("n,m,reg", SHAPES)
def test_fused_bcd_matches_oracle(gpu_lib, n, m, reg):
    M, a, b = cloud_problem(n, m, seed=n + m)
    M32 = M.astype(np.float32)
    print("fused bcd %dx%d reg=%g" % (n, m, reg), flush=True)
    r, nf = solve(gpu_lib, M32, a, b, reg, 1e-8, 5000, fused=1)
    o = O.sinkhorn_bcd(M32.astype(np.float64), a, b, reg, tol=1e-8, max_iter=5000)
    assert nf == fused_expected(r)    # every FP32 iteration used the single read
    assert r.niter < 5000 and abs(r.niter - o["niter"]) <= max(2, 0.02 * o["niter"])
    assert len(r.obj_vals) == r.niter + 1
    assert r.mar_errs[-1] < 1e-8 and all(e >= 1e-8 for e in r.mar_errs[:-1])
    k = min(10, len(o["obj_vals"]), len(r.obj_vals))
    np.testing.assert_allclose(r.obj_vals[:k], o["obj_vals"][:k], rtol=1e-9)
    assert rel_err(r.dual, o["dual"]) < 1e-6
    assert r.mar_err_fp64 < 1.05e-8


def test_fused_matches_two_pass(gpu_lib):
    M, a, b = cloud_problem(400, 9000, seed=4)
    M32 = M.astype(np.float32)
    print("fused vs two-pass 400x9000", flush=True)
    rf, nf = solve(gpu_lib, M32, a, b, 0.02, 1e-8, 5000, fused=1)
    rt, nt = solve(gpu_lib, M32, a, b, 0.02, 1e-8, 5000, fused=0)
    assert nf > 0 and nt == 0
    assert abs(rf.niter - rt.niter) <= 1
    assert abs(rf.obj_fp64 - rt.obj_fp64) < 1e-12 * abs(rt.obj_fp64)
    assert rel_err(rf.dual, rt.dual) < 1e-7
    assert rf.mar_err_fp64 < 1.05e-8 and rt.mar_err_fp64 < 1.05e-8


def test_fused_row_range_fallback(gpu_lib):
    # Row 0 is free (M = 0) but carries a_0 = 1e-7: in the first iteration its
    # row sum is ~1e7 a_0.  Row 1 costs 1 everywhere at reg 0.01: its terms
    # are ~2^-144, below FP32 range.  Both rows leave [2^-20, 2^20] and take
    # the exact-maximum path.
    n, m, reg = 40, 3000, 0.01
    M, a, b = cloud_problem(n, m, seed=21)
    M[0, :] = 0.0
    M[1, :] = 1.0
    a[0] = 1e-7
    a /= a.sum()
    M32 = M.astype(np.float32)
    print("fused bcd range fallback", flush=True)
    r, nf = solve(gpu_lib, M32, a, b, reg, 1e-6, 20000, fused=1)
    o = O.sinkhorn_bcd(M32.astype(np.float64), a, b, reg, tol=1e-6, max_iter=20000)
    assert nf > 0 and np.all(np.isfinite(r.dual))
    assert abs(r.niter - o["niter"]) <= max(2, 0.02 * o["niter"])
    # the in-loop objective sums FP32 terms: ~1e-7 relative of reg sum r
    np.testing.assert_allclose(r.obj_vals[:5], o["obj_vals"][:5], rtol=0, atol=1e-7 * reg)
    assert rel_err(r.dual, o["dual"]) < 1e-6
    assert r.mar_err_fp64 < 1.05e-6


def test_fused_warm_start(gpu_lib):
    # with x0 the first iteration keeps the two-pass form (its beta is not
    # the result of a beta update), the rest run single-read
    M, a, b = cloud_problem(200, 6000, seed=5)
    M32 = M.astype(np.float32)
    r0, _ = solve(gpu_lib, M32, a, b, 0.03, 1e-3, 5, fused=0)
    x0 = np.asarray(r0.dual) + 0.01
    rf, nf = solve(gpu_lib, M32, a, b, 0.03, 1e-8, 5000, fused=1, x0=x0)
    rt, _ = solve(gpu_lib, M32, a, b, 0.03, 1e-8, 5000, fused=0, x0=x0)
    assert nf == rf.niter           # all but iteration 0
    assert abs(rf.niter - rt.niter) <= 1 and rel_err(rf.dual, rt.dual) < 1e-7
    assert rf.mar_err_fp64 < 1.05e-8


def test_fused_ineligible_marginals_fall_back(gpu_lib):
    # min a min b below 2^-60 sum a sum b: the single-read pass is not used,
    # and the result is the two-pass one bit for bit
    M, a, b = cloud_problem(100, 3000, seed=6)
    a[3] = 1e-40
    a /= a.sum()
    M32 = M.astype(np.float32)
    rf, nf = solve(gpu_lib, M32, a, b, 0.05, 1e-8, 5000, fused=1)
    rt, _ = solve(gpu_lib, M32, a, b, 0.05, 1e-8, 5000, fused=0)
    assert nf == 0
    assert rf.niter == rt.niter and np.array_equal(rf.dual, rt.dual)


def test_fused_many_rows_per_workgroup(gpu_lib):
    # 140000 rows over at most 256 workgroups: > 512 rows each, more rows than
    # threads, so every thread finishes several rows in the epilogue
    n, m, reg = 140000, 1100, 0.05
    rng = np.random.default_rng(7)
    X = rng.standard_normal((n, 8)).astype(np.float32)
    Y = rng.standard_normal((m, 8)).astype(np.float32)
    M = (X * X).sum(1)[:, None] + (Y * Y).sum(1)[None, :] - 2.0 * (X @ Y.T)
    np.maximum(M, 0.0, out=M)
    M /= M.max()
    a = 0.9 * rng.dirichlet(np.ones(n)) + 0.1 / n
    b = 0.9 * rng.dirichlet(np.ones(m)) + 0.1 / m
    a /= a.sum()
    b /= b.sum()
    print("fused bcd 140000x1100", flush=True)
    rf, nf = solve(gpu_lib, M, a, b, reg, 1e-7, 2000, fused=1)
    rt, _ = solve(gpu_lib, M, a, b, reg, 1e-7, 2000, fused=0)
    assert nf == rf.niter + 1
    assert abs(rf.niter - rt.niter) <= 1
    assert rel_err(rf.dual, rt.dual) < 1e-6
    assert rf.mar_err_fp64 < 1.05e-7


def test_fused_edge_shapes(gpu_lib):
    # one row; three rows over the full 16384 columns (one row per workgroup);
    # max_iter = 0 and an immediately met tolerance: the single-read pass
    # still runs the stop test of iteration 0.  (Rows carry a_i ~ 1 / n here:
    # FP32-bulk row sums resolve their marginal to ~1e-7, hence tol 1e-6.)
    for n, m in ((1, 3000), (3, 16384)):
        M, a, b = cloud_problem(n, m, seed=n)
        M32 = M.astype(np.float32)
        print("fused edge %dx%d" % (n, m), flush=True)
        r, nf = solve(gpu_lib, M32, a, b, 0.05, 1e-6, 200, fused=1)
        o = O.sinkhorn_bcd(M32.astype(np.float64), a, b, 0.05, tol=1e-6, max_iter=200)
        assert nf == r.niter + 1 and abs(r.niter - o["niter"]) <= 1
        assert rel_err(r.dual, o["dual"]) < 1e-6
    M, a, b = cloud_problem(50, 2500, seed=3)
    M32 = M.astype(np.float32)
    for tol, max_iter in ((1e-8, 0), (1e9, 100)):
        r, nf = solve(gpu_lib, M32, a, b, 0.05, tol, max_iter, fused=1)
        o = O.sinkhorn_bcd(M32.astype(np.float64), a, b, 0.05, tol=tol, max_iter=max_iter)
        assert r.niter == o["niter"] == 0 and nf == 1 and len(r.obj_vals) == 1
        np.testing.assert_allclose(r.obj_vals, o["obj_vals"], rtol=1e-9)
        assert rel_err(r.dual, o["dual"]) < 1e-6


@pytest.mark.parametrize("n,m,reg,tol,uniform", [(1, 3000, 0.05, 1e-9, False),
                                                 (3, 16384, 0.05, 1e-9, False),
                                                 (50, 2500, 0.05, 1e-10, False),
                                                 (1200, 1100, 0.01, 1e-10, True)])
def test_fp32_bulk_finishes_below_its_resolution(gpu_lib, n, m, reg, tol, uniform):
    # FP32 sums resolve each marginal to ~2^-23 of its size; below that the
    # FP32 loop hands over to FP64 passes over the same FP32 M and goes on to
    # tol, so the iteration count and the dual match the FP64 oracle's.
    M, a, b = cloud_problem(n, m, d=4 if uniform else 16, seed=n + 3)
    if uniform:
        a, b = np.full(n, 1.0 / n), np.full(m, 1.0 / m)
    M32 = M.astype(np.float32)
    print("fp32 finish %dx%d tol %g" % (n, m, tol), flush=True)
    r, nf = solve(gpu_lib, M32, a, b, reg, tol, 5000, fused=1)
    o = O.sinkhorn_bcd(M32.astype(np.float64), a, b, reg, tol=tol, max_iter=5000)
    pf = r.stats["precise_from"]
    assert 0 <= pf <= r.niter and nf == fused_expected(r)
    assert abs(r.niter - o["niter"]) <= 1
    assert r.mar_errs[-1] < tol and r.mar_err_fp64 < 1.05 * tol
    assert len(r.obj_vals) == len(r.mar_errs) == len(r.run_times) == r.niter + 1
    assert all(e >= tol for e in r.mar_errs[:-1])
    # FP32-bulk objectives carry ~1e-9 relative sum error; from the handover
    # on they are FP64 sums along a trajectory within ~1e-8 of the oracle's
    k = min(len(r.obj_vals), len(o["obj_vals"]))
    np.testing.assert_allclose(r.obj_vals[:k], o["obj_vals"][:k], rtol=1e-8)
    np.testing.assert_allclose(r.obj_vals[pf:k], o["obj_vals"][pf:k], rtol=1e-11)
    assert rel_err(r.dual, o["dual"]) < 1e-8


# --- several rows per step (m <= 8192, FP32 and FP64 arithmetic) ---------------

def fixed_iterations(gpu_lib, M, a, b, reg, iters, bulk, fused=1):
    """The iterates of a fixed number of iterations and the passes that ran:
    (result, FP32 single-read passes, FP64 single-read passes)."""
    with gpu_lib.Problem(M, a, b, reg, bulk=bulk) as P:
        P.profile(True)
        r = P.solve(0, tol=0.0, max_iter=iters, compute_plan=False, bcd_fused=fused)
        return r, P.profile_stats(2)[0], P.profile_stats(4)[0]


# FP64: one thread per 2 columns, 512 threads: NC = ceil(m / 1024); 256 threads
# up to m = 512.  Rows per workgroup from 1 to 79 (more than one wave's lanes).
@pytest.mark.parametrize("n,m", [(1, 1), (7, 2), (300, 80), (50, 511), (50, 512), (700, 513),
                                 (40, 1024), (1030, 1025), (70, 2049), (260, 3073), (33, 4096),
                                 (33, 5121), (9, 6145), (300, 7169), (5, 8192), (20000, 20),
                                 (10, 8193)])
def test_fp64_single_read_iterates(gpu_lib, n, m):
    # The iterates are those of the oracle's FP64 iteration; sums run in
    # another order: a relative 1e-15 per sum and step, 12 steps.
    M, a, b = cloud_problem(n, m, seed=n + m)
    reg = 0.03
    print("fp64 single read %dx%d" % (n, m), flush=True)
    r, _, passes = fixed_iterations(gpu_lib, M, a, b, reg, 12, "fp64")
    assert passes == (13 if m <= 8192 else 0) and r.niter == 12
    o = O.sinkhorn_bcd(M, a, b, reg, tol=0.0, max_iter=12)
    assert rel_err(r.dual, o["dual"]) < 1e-12
    np.testing.assert_allclose(r.obj_vals, o["obj_vals"], rtol=1e-11, atol=1e-15)
    np.testing.assert_allclose(r.mar_errs, o["mar_errs"], rtol=1e-7, atol=1e-14)


@pytest.mark.parametrize("n,m", [(1, 1), (300, 80), (1300, 1024), (40, 1025), (520, 2047),
                                 (1025, 4096), (11, 6143), (600, 8192)])
def test_fp32_single_read_iterates(gpu_lib, n, m):
    # FP32 terms: 2^-24 per exponential and per product, sums of FP32 partials
    M, a, b = cloud_problem(n, m, seed=n + m, dtype=np.float32)
    reg = 0.05
    print("fp32 single read %dx%d" % (n, m), flush=True)
    tol_floor = 0.5 * 2.0 ** -22 * np.sqrt((a * a).sum() + (b * b).sum())
    with gpu_lib.Problem(M, a, b, reg) as P:
        P.profile(True)
        r = P.solve(0, tol=2 * tol_floor, max_iter=5, compute_plan=False)
        passes = P.profile_stats(2)[0]
    o = O.sinkhorn_bcd(M.astype(np.float64), a, b, reg, tol=0.0, max_iter=r.niter)
    assert passes == r.niter + 1
    assert rel_err(r.dual, o["dual"]) < 1e-6


@pytest.mark.parametrize("m", [700, 1024, 1025, 3000, 5000, 8000])
def test_fp64_finish_runs_single_read(gpu_lib, m):
    # an FP32 solve below its resolution: the FP64 finish reads M once per
    # iteration too, and reaches the oracle's iterate
    n, reg, tol = 90, 0.05, 1e-11
    M, a, b = cloud_problem(n, m, seed=m, dtype=np.float32)
    print("fp64 finish m=%d" % m, flush=True)
    with gpu_lib.Problem(M, a, b, reg) as P:
        P.profile(True)
        r = P.solve(0, tol=tol, max_iter=2000, compute_plan=False, verify=True)
        fine = P.profile_stats(4)[0]
    pf = r.stats["precise_from"]
    o = O.sinkhorn_bcd(M.astype(np.float64), a, b, reg, tol=tol, max_iter=2000)
    assert pf >= 0 and fine == r.niter - pf + 1
    assert r.mar_err_fp64 < 1.05 * tol and abs(r.niter - o["niter"]) <= 1
    assert rel_err(r.dual, o["dual"]) < 1e-10


def test_fp64_row_range_fallback(gpu_lib):
    # at reg 1e-4 the terms span 2^-14000: rows leave [2^-400, 2^400] at first
    n, m, reg = 70, 900, 1e-4
    M, a, b = cloud_problem(n, m, seed=2)
    M[0, :] = 0.0
    M[1, :] = 1.0
    a[0] = 1e-7
    a /= a.sum()
    print("fp64 range fallback", flush=True)
    r, _, passes = fixed_iterations(gpu_lib, M, a, b, reg, 20, "fp64")
    t, _, none = fixed_iterations(gpu_lib, M, a, b, reg, 20, "fp64", fused=0)
    assert passes == 21 and none == 0 and np.all(np.isfinite(r.dual))
    o = O.sinkhorn_bcd(M, a, b, reg, tol=0.0, max_iter=20)
    # arguments of 1e4 carry 1e-12 absolute: duals to reg times that and more
    assert rel_err(r.dual, o["dual"]) < 1e-11 and rel_err(t.dual, o["dual"]) < 1e-11
    np.testing.assert_allclose(r.mar_errs, o["mar_errs"], rtol=1e-6, atol=1e-12)


# --- infinite costs and non-finite warm starts -----------------------------------

# one and several rows per workgroup, the step's last rows repeated or not
@pytest.mark.parametrize("bulk,n,m", [("fp64", 30, 20), ("fp64", 300, 33), ("fp64", 30, 3000),
                                      ("fp32", 60, 700), ("fp32", 1030, 700), ("fp32", 30, 3000),
                                      ("fp32", 700, 5000)])
def test_single_read_row_without_finite_cost(gpu_lib, bulk, n, m):
    # a row of infinite costs has no mass to give: its potential is +inf and the
    # others' iterates are those of the problem without it
    M, a, b = cloud_problem(n, m, seed=n + m)
    M = M.astype(np.float32 if bulk == "fp32" else np.float64)
    for row in (n // 2, n - 1):
        M2 = M.copy()
        M2[row, :] = np.inf
        print("infinite row %d of %dx%d %s" % (row, n, m, bulk), flush=True)
        r, f32, f64 = fixed_iterations(gpu_lib, M2, a, b, 0.05, 4, bulk)
        assert f32 + f64 == 5 and r.niter == 4
        keep = np.arange(n) != row
        o = O.sinkhorn_bcd(M[keep].astype(np.float64), a[keep], b, 0.05, tol=0.0, max_iter=4)
        assert r.dual[row] == np.inf
        assert rel_err(np.delete(r.dual, row), o["dual"]) < (1e-6 if bulk == "fp32" else 1e-12)


@pytest.mark.parametrize("bulk,n,m", [("fp64", 30, 20), ("fp64", 30, 3000), ("fp32", 60, 700),
                                      ("fp32", 30, 3000), ("fp32", 1030, 3000)])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_single_read_recovers_from_a_warm_start(gpu_lib, bulk, n, m, bad):
    # alpha_0 only guesses the scale of the first row sums; a row whose guess is
    # not finite is formed again by the next iteration
    M, a, b = cloud_problem(n, m, seed=n + m)
    M = M.astype(np.float32 if bulk == "fp32" else np.float64)
    x0 = 0.01 * np.random.default_rng(3).standard_normal(n + m - 1)
    x0[n - 1] = bad
    print("warm start with %s %dx%d %s" % (bad, n, m, bulk), flush=True)
    with gpu_lib.Problem(M, a, b, 0.05, bulk=bulk) as P:
        r = P.solve(0, tol=1e-8, max_iter=2000, compute_plan=False, x0=x0)
        c = P.solve(0, tol=1e-8, max_iter=2000, compute_plan=False)
    assert r.niter < 2000 and np.all(np.isfinite(r.dual))
    assert rel_err(r.dual, c.dual) < 1e-5      # both within tol of the one solution


# four and sixteen threads per column in the combine (4 and 5 row blocks of 16),
# and 64- and 16-column workgroups with a remainder; 131101 columns: 513 tiles of
# 256 and so one row block, and more tile sums than eight per thread
@pytest.mark.parametrize("n,m", [(64, 65), (65, 65), (64, 1007), (65, 1007), (3, 1), (70, 16),
                                 (17, 131101)])
@pytest.mark.parametrize("bulk", ["fp32", "fp64"])
def test_two_pass_combine_splits(gpu_lib, bulk, n, m):
    M, a, b = cloud_problem(n, m, d=4, seed=n + m)
    M = M.astype(np.float32 if bulk == "fp32" else np.float64)
    print("two-pass combine %dx%d %s" % (n, m, bulk), flush=True)
    r, f32, f64 = fixed_iterations(gpu_lib, M, a, b, 0.05, 4, bulk, fused=0)
    assert (f32, f64) == (0, 0)
    o = O.sinkhorn_bcd(M.astype(np.float64), a, b, 0.05, tol=0.0, max_iter=4)
    assert rel_err(r.dual, o["dual"]) < (1e-6 if bulk == "fp32" else 1e-12)
    np.testing.assert_allclose(r.obj_vals, o["obj_vals"], rtol=1e-7 if bulk == "fp32" else 1e-11)
    # FP64: the sums of squares over all tiles; FP32 rounds each row sum to 2^-23
    np.testing.assert_allclose(r.mar_errs, o["mar_errs"], rtol=1e-2 if bulk == "fp32" else 1e-7,
                               atol=2e-7 if bulk == "fp32" else 1e-14)


# --- tall, narrow matrices -------------------------------------------------------

# (bulk, m, rows per compute unit, single read): the strips of the two-pass form
# are 256 (FP32) and 128 (FP64) columns wide; one or two strips and more than 192
# (FP64 arithmetic: 128) rows per unit and strip take two passes
@pytest.mark.parametrize("bulk,m,rows,single", [
    ("fp32", 40, 192, True), ("fp32", 40, 193, False), ("fp32", 256, 200, False),
    ("fp32", 257, 384, True), ("fp32", 257, 385, False), ("fp32", 513, 400, True),
    ("fp64", 40, 128, True), ("fp64", 40, 129, False), ("fp64", 129, 256, True),
    ("fp64", 129, 257, False), ("fp64", 257, 300, True)])
def test_tall_narrow_form(gpu_lib, bulk, m, rows, single):
    import torch
    n = rows * torch.cuda.get_device_properties(0).multi_processor_count
    rng = np.random.default_rng(m)
    x, y = rng.random((n, 1)), rng.random((1, m))
    M = ((x - y) ** 2).astype(np.float32 if bulk == "fp32" else np.float64)
    a, b = np.full(n, 1.0 / n), np.full(m, 1.0 / m)
    print("tall %dx%d %s" % (n, m, bulk), flush=True)
    with gpu_lib.Problem(M, a, b, 0.05, bulk=bulk) as P:
        P.profile(True)
        r = P.solve(0, tol=0.0 if bulk == "fp64" else 1e-6, max_iter=3, compute_plan=False)
        one, two = P.profile_stats(2 if bulk == "fp32" else 4)[0], P.profile_stats(0)[0]
    assert (one, two) == ((r.niter + 1, 0) if single else (0, r.niter + 1))
    o = O.sinkhorn_bcd(M.astype(np.float64), a, b, 0.05, tol=0.0, max_iter=r.niter)
    assert rel_err(r.dual, o["dual"]) < (1e-6 if bulk == "fp32" else 1e-12)


def test_tall_narrow_fp64_finish(gpu_lib):
    # between the two limits: FP32 iterations in one read, their FP64 finish in two
    import torch
    n, m = 160 * torch.cuda.get_device_properties(0).multi_processor_count, 40
    rng = np.random.default_rng(m)
    M = ((rng.random((n, 1)) - rng.random((1, m))) ** 2).astype(np.float32)
    a, b = np.full(n, 1.0 / n), np.full(m, 1.0 / m)
    with gpu_lib.Problem(M, a, b, 0.05) as P:
        P.profile(True)
        r = P.solve(0, tol=1e-12, max_iter=2000, compute_plan=False, verify=True)
        counts = [P.profile_stats(k)[0] for k in (0, 2, 4)]
    pf = r.stats["precise_from"]
    assert pf >= 0 and counts == [r.niter - pf + 1, pf + 1, 0]
    assert r.mar_err_fp64 < 1.05e-12
