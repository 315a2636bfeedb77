"""GPU parity of the dense CP adapter's forward (purin_cp_dense_solve) with the
oracle (oracle/dense.py: solve_dense, chambolle_pock/dense.py:26-105 -- factored
prox, no freezing, no stationarity test, power-iteration steps), through the C
ABI.  The oracle is pinned in tests/test_oracle_dense.py."""

import numpy as np
import pytest

from oracle import dense as od
from tests._gpu import rel_err, require_gpu, to_np

pytestmark = pytest.mark.gpu

TOL = {np.float64: 1e-10, np.float32: 1e-4}


def _dense_plan(n, me, mi, dtype, support=None, **kw):
    import torch
    from purin_amd.plan import Plan

    rows = [list(range(n))] * me + ([list(range(n))] * mi if support is None else
                                    [sorted(r) for r in support])
    indptr = np.zeros(len(rows) + 1, np.int64)
    indptr[1:] = np.cumsum([len(r) for r in rows])
    indices = np.asarray([c for r in rows for c in r], np.int32)
    return Plan(n, me, mi, indptr, indices, np.ones(indptr[-1]),
                dtype=torch.float64 if dtype == np.float64 else torch.float32,
                bound_presolve=False, row_scaling=False, norm_bound=False, device="cuda", **kw)


def _problem(seed, B=24, n=12, me=3, mi=5):
    rng = np.random.default_rng(seed)
    q = rng.uniform(0.5, 3.0, (B, n))
    c = rng.normal(size=(B, n))
    A = rng.normal(size=(B, me, n))
    C = rng.normal(size=(B, mi, n))
    x0 = rng.uniform(-0.3, 0.3, (B, n))
    b = np.einsum("bmn,bn->bm", A, x0)
    d = np.einsum("bmn,bn->bm", C, x0) + rng.uniform(0.1, 0.5, (B, mi))
    lo, hi = np.full((B, n), -1.0), np.full((B, n), 1.0)
    return q, c, A, b, C, d, lo, hi


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("accelerated", [False, True])
@pytest.mark.parametrize("early_stop", [False, True])
def test_dense_solve_matches_oracle(dtype, accelerated, early_stop):
    require_gpu()
    q, c, A, b, C, d, lo, hi = (x.astype(dtype) for x in _problem(51))
    B, n = q.shape
    me, mi = A.shape[1], C.shape[1]
    iters = 400
    tol = (1e-7 if dtype == np.float64 else 1e-3) if early_stop else 0.0
    y, lam, mu, it, _ = od.solve_dense(q, c, A, b, C, d, lo, hi, accelerated=accelerated,
                                       max_iterations=iters, tolerance=max(tol, 1e-300))
    plan = _dense_plan(n, me, mi, dtype, accelerated=accelerated)
    values = np.concatenate((A, C), axis=1).reshape(B, -1)
    gy, gm, git, _ = plan.dense_solve(q, c, np.concatenate((b, d), axis=1), lo, hi, values=values,
                                      tolerance=max(tol, 1e-30), max_iterations=iters,
                                      early_stop=early_stop, check_every=7)
    # no freezing: every sample runs until the last one is accepted
    np.testing.assert_array_equal(to_np(git), it)
    assert len(np.unique(it)) == 1
    if early_stop and dtype == np.float64 and not accelerated:
        assert it[0] < iters  # the stop test fired (accelerated fp64 stalls above 1e-7)
    assert rel_err(to_np(gy), y) <= TOL[dtype]
    assert rel_err(to_np(gm), np.concatenate((lam, mu), axis=1)) <= TOL[dtype]


@pytest.mark.parametrize("n,me,mi,B,accelerated,dtype", [
    (7, 1, 1, 3, False, np.float64),      # one lane per row and column
    (13, 2, 3, 5, True, np.float64),      # two lanes per row
    (60, 12, 25, 7, False, np.float64),   # eight and four lanes
    (60, 12, 25, 7, True, np.float64),
    (120, 20, 44, 4, False, np.float64),  # sixteen wavefronts: none left for the stop test
    (150, 10, 21, 3, False, np.float32),
    (200, 20, 44, 2, False, np.float64),  # too large for the one-workgroup loop
])
def test_dense_one_workgroup_loop(n, me, mi, B, accelerated, dtype):
    """Lanes per row and column, wavefront counts and the two launches (to each sample's own
    acceptance, then to the last one's) against the oracle; fixed iterations too."""
    require_gpu()
    q, c, A, b, C, d, lo, hi = (x.astype(dtype) for x in _problem(61, B=B, n=n, me=me, mi=mi))
    plan = _dense_plan(n, me, mi, dtype, accelerated=accelerated)
    values = np.concatenate((A, C), axis=1).reshape(B, -1)
    tol = (1e-4 if accelerated else 1e-6) if dtype == np.float64 else 1e-2
    for early, iters, t in ((True, 3000, tol), (False, 60, 1e-30)):
        y, lam, mu, it, _ = od.solve_dense(q, c, A, b, C, d, lo, hi, accelerated=accelerated,
                                           max_iterations=iters, tolerance=max(t, 1e-300))
        gy, gm, git, _ = plan.dense_solve(q, c, np.concatenate((b, d), axis=1), lo, hi,
                                          values=values, tolerance=t, max_iterations=iters,
                                          early_stop=early)
        if dtype == np.float64:
            np.testing.assert_array_equal(to_np(git), it)
            assert rel_err(to_np(gy), y) <= TOL[dtype]
            assert rel_err(to_np(gm), np.concatenate((lam, mu), axis=1)) <= TOL[dtype]
        else:  # a stop a few iterations away moves the iterate by the tolerance at most
            assert abs(int(to_np(git)[0]) - int(it[0])) <= 0.1 * int(it[0])
            assert rel_err(to_np(gy), y) <= (5 * tol if early else TOL[dtype])
        if early:
            assert it[0] < iters


@pytest.mark.parametrize("n,me,mi", [(13, 2, 3), (60, 12, 25), (200, 20, 44)])
@pytest.mark.parametrize("early", [False, True])
def test_dense_nonfinite_inputs(n, me, mi, early):
    """A NaN bound, a NaN and an infinite cost and infinite bounds, each in one sample: non-finite
    entries in the oracle's places, the other samples at the parity bar.  A sample with a
    non-finite iterate is never accepted, so every sample runs to the limit."""
    require_gpu()
    q, c, A, b, C, d, lo, hi = _problem(62, B=6, n=n, me=me, mi=mi)
    lo[1, 2] = np.nan
    c[2, 3] = np.nan
    c[3, 1] = -np.inf
    lo[4], hi[4] = -np.inf, np.inf
    iters = 40
    with np.errstate(invalid="ignore", over="ignore"):
        y, lam, mu, it, _ = od.solve_dense(q, c, A, b, C, d, lo, hi, max_iterations=iters,
                                           tolerance=1e-3 if early else 1e-300)
    want, wm = y, np.concatenate((lam, mu), axis=1)
    assert np.all(it == iters) and not np.isfinite(y[[1, 2]]).all(axis=1).any()
    got, gm, git, _ = _dense_plan(n, me, mi, np.float64).dense_solve(
        q, c, np.concatenate((b, d), axis=1), lo, hi,
        values=np.concatenate((A, C), axis=1).reshape(6, -1), max_iterations=iters,
        tolerance=1e-3 if early else 1e-30, early_stop=early)
    np.testing.assert_array_equal(to_np(git), it)
    for g, w in ((to_np(got), want), (to_np(gm), wm)):
        np.testing.assert_array_equal(np.isnan(g), np.isnan(w))
        inf = np.isinf(w)
        np.testing.assert_array_equal(np.isinf(g), inf)
        np.testing.assert_array_equal(g[inf], w[inf])
        fin = np.isfinite(w)
        assert rel_err(g[fin], w[fin]) <= TOL[np.float64]


def test_dense_packed_inequality_support():
    """A packed inequality support (sparse_layer.py:44-122): the inequality rows
    keep only their listed columns; the same iteration otherwise."""
    require_gpu()
    q, c, A, b, C, d, lo, hi = _problem(52, B=16, n=10, me=2, mi=4)
    support = [[0, 3, 4], [1, 2], [5, 6, 7, 9], [8]]
    mask = np.zeros(C.shape[1:], bool)
    for i, r in enumerate(support):
        mask[i, r] = True
    C = np.where(mask[None], C, 0.0)
    x0 = np.zeros((16, 10))
    d = np.abs(d)
    y, lam, mu, it, _ = od.solve_dense(q, c, A, b, C, d, lo, hi, max_iterations=300,
                                       tolerance=1e-300)
    plan = _dense_plan(10, 2, 4, np.float64, support=support)
    packed = np.concatenate((A.reshape(16, -1), C[:, mask]), axis=1)
    gy, gm, git, _ = plan.dense_solve(q, c, np.concatenate((b, d), axis=1), lo, hi,
                                      values=packed, max_iterations=300, early_stop=False)
    assert rel_err(to_np(gy), y) <= 1e-10
    assert rel_err(to_np(gm), np.concatenate((lam, mu), axis=1)) <= 1e-9


def test_dense_known_answer_and_warm_start():
    """Reference tests/test_dense_cp.py:20-45: [1/3, 2/3] and warm start."""
    require_gpu()
    plan = _dense_plan(2, 1, 1, np.float64)
    q, c = np.array([[2.0, 4.0]]), np.array([[-2.0, -4.0]])
    vals = np.array([[1.0, 1.0, -1.0, 0.0]])
    rhs = np.array([[1.0, 0.0]])
    lo, hi = np.zeros((1, 2)), np.full((1, 2), 2.0)
    for accelerated in (False, True):
        plan = _dense_plan(2, 1, 1, np.float64, accelerated=accelerated)
        y, m, it, _ = plan.dense_solve(q, c, rhs, lo, hi, values=vals, tolerance=1e-13,
                                       max_iterations=20000)
        np.testing.assert_allclose(to_np(y), [[1 / 3, 2 / 3]], atol=1e-6)
        w, _, _, _ = plan.dense_solve(q, c, rhs, lo, hi, values=vals, y0=y, dual0=m,
                                      tolerance=1e-13, max_iterations=20000)
        np.testing.assert_allclose(to_np(w), to_np(y), atol=1e-6)


@pytest.mark.parametrize("with_dual_cotangent", [False, True])
@pytest.mark.parametrize("tol,iters,bar", [(1e-6, 50, 1e-5), (1e-12, 400, 1e-9)])
def test_dense_adjoint_matches_oracle_at_the_same_state(with_dual_cotangent, tol, iters, bar):
    """BiCGSTAB over the batch with the frozen prox (dense_implicit.py:160-210) at
    the GPU's state, with the same iteration count.  Converged (1e-12) the
    gradients agree to 1e-9; at the reference's 1e-6 the unconverged iterate
    depends on the rounding of the global dot products (summed in another
    order), and agrees to 10 x that tolerance.  The iteration counts agree to
    two (the last stop test moves with the operator's rounding)."""
    require_gpu()
    q, c, A, b, C, d, lo, hi = _problem(53, B=8, n=10, me=2, mi=4)
    B, n = q.shape
    me, mi = 2, 4
    plan = _dense_plan(n, me, mi, np.float64)
    values = np.concatenate((A, C), axis=1)
    rhs = np.concatenate((b, d), axis=1)
    y, m, it, saved = plan.dense_solve(q, c, rhs, lo, hi, values=values.reshape(B, -1),
                                       tolerance=1e-10, max_iterations=20000, save=True)
    rng = np.random.default_rng(4)
    cot = rng.normal(size=(B, n))
    cotd = rng.normal(size=(B, me + mi)) if with_dual_cotangent else np.zeros((B, me + mi))
    want = od.implicit_vjp(q, c, values, rhs, lo, hi, me, to_np(y), to_np(m), cot, cotd,
                           tolerance=tol, adjoint_iterations=iters)
    got = plan.dense_adjoint(saved, q, c, cot, values=values.reshape(B, -1),
                             cot_dual=cotd if with_dual_cotangent else None, tolerance=tol,
                             max_iterations=iters)
    stats = plan.last_adjoint_stats()
    # the first iteration under the stop threshold moves with the operator's
    # rounding: with unit-roundoff noise on each operator output the oracle's
    # own count spans 59-61 here (10 noise seeds, tolerance 1e-12)
    assert abs(stats["arnoldi_steps"] - want[5]) <= 2 and want[5] > 0
    np.testing.assert_array_equal(to_np(got.g_q), 0.0)
    for name, w in (("g_c", want[0]), ("g_values", want[1].reshape(B, -1)), ("g_rhs", want[2]),
                    ("g_lower", want[3]), ("g_upper", want[4])):
        assert rel_err(to_np(getattr(got, name)), w) <= bar, name


@pytest.mark.parametrize("n,me,mi,B", [
    (60, 12, 25, 5),    # four wavefronts sharing a slice of rows and of columns
    (100, 30, 70, 66),  # two slices each
    (230, 20, 40, 3),   # eight wavefronts
    (8, 2, 3, 1030),    # more samples than take a workgroup each: the batch-minor passes
])
def test_dense_adjoint_wide_rows(n, me, mi, B):
    """The per-sample BiCGSTAB kernels where wavefronts share a slice's entries, at the
    GPU's state and converged: the solution is fixed to the residual (1e-12) times the
    system's condition, below 1e4 here."""
    require_gpu()
    q, c, A, b, C, d, lo, hi = _problem(71, B=B, n=n, me=me, mi=mi)
    plan = _dense_plan(n, me, mi, np.float64)
    values = np.concatenate((A, C), axis=1)
    rhs = np.concatenate((b, d), axis=1)
    y, m, it, saved = plan.dense_solve(q, c, rhs, lo, hi, values=values.reshape(B, -1),
                                       tolerance=1e-6, max_iterations=20000, save=True)
    cot = np.random.default_rng(5).normal(size=(B, n))
    cotd = np.zeros((B, me + mi))
    want = od.implicit_vjp(q, c, values, rhs, lo, hi, me, to_np(y), to_np(m), cot, cotd,
                           tolerance=1e-12, adjoint_iterations=2000)
    got = plan.dense_adjoint(saved, q, c, cot, values=values.reshape(B, -1), tolerance=1e-12,
                             max_iterations=2000)
    assert 0 < want[5] < 2000 and 0 < plan.last_adjoint_stats()["cycles"] < 2000
    for name, w in (("g_c", want[0]), ("g_values", want[1].reshape(B, -1)), ("g_rhs", want[2])):
        assert rel_err(to_np(getattr(got, name)), w) <= 1e-8, name
