"""The CP loop with one workgroup per sample (solo.hip) at the edges of its dispatch:
wavefront counts with and without the wavefront of the stop test, idle wavefronts, rows
and columns wider than the entries held in registers, and the batches where the tile
kernels take over.  Held to the streaming passes on the whole batch, whose sums run in
another order: the bars of the resident kernels' tests (fp64 counts identical; in fp32 a
stop may fall elsewhere in at most 1 of 10 samples)."""

import numpy as np
import pytest

from purin_amd import workloads
from tests._gpu import canonical_from_workload, plan_for, rel_err, require_gpu, to_np

pytestmark = pytest.mark.gpu

TOL = {np.float64: 1e-10, np.float32: 1e-4}


@pytest.mark.parametrize("n,me,mi,wmin,wmax,B,dtype", [
    (64, 10, 20, 2, 9, 5, np.float64),       # one wavefront of columns; columns past 8 entries
    (65, 10, 20, 2, 12, 5, np.float64),      # two; rows past 8 entries
    (40, 30, 170, 2, 4, 3, np.float64),      # more rows than columns, wide columns
    (250, 40, 60, 2, 6, 512, np.float64),    # four wavefronts, padded to seven and the test's
    (250, 40, 60, 2, 6, 513, np.float64),    # four without the test's wavefront
    (330, 40, 60, 2, 6, 9, np.float64),      # six, padded
    (500, 40, 60, 2, 6, 256, np.float64),    # eight with the test's wavefront
    (500, 40, 60, 2, 6, 257, np.float64),    # eight without
    (600, 60, 150, 2, 6, 257, np.float64),   # ten: fixed iterations go to the tiles
    (960, 90, 200, 2, 6, 7, np.float64),     # fifteen and the test's
    (961, 90, 200, 2, 6, 7, np.float64),     # sixteen
    (900, 90, 200, 2, 6, 300, np.float64),   # fifteen: the tiles
    (1024, 100, 924, 2, 5, 4, np.float64),   # the largest
    (200, 30, 60, 2, 7, 70, np.float32),
    (600, 60, 150, 2, 6, 600, np.float32),   # fixed iterations on the tiles
    (600, 60, 150, 2, 6, 800, np.float32),   # both loops on the tiles
])
@pytest.mark.parametrize("accelerated", [False, True])
def test_solo_matches_streaming(n, me, mi, wmin, wmax, B, dtype, accelerated):
    require_gpu()
    w = workloads.ragged_rows(700 + n, n=n, me=me, mi=mi, wmin=wmin, wmax=wmax, batch=B,
                              accelerated=accelerated)
    canon = canonical_from_workload(w)
    plan = plan_for(canon, dtype=dtype, accelerated=accelerated)
    rhs = np.tile(w.rhs, (B, 1)).astype(dtype)
    target = w.target.astype(dtype)
    bar = TOL[dtype]
    # bounds shared, and scaled per sample (their rows are the last 2 n)
    scaled = rhs.copy()
    scaled[:, me + mi:] *= np.linspace(0.8, 1.2, B).astype(dtype)[:, None]
    for r, shared in ((rhs, True), (scaled, False)):
        kw = dict(max_iterations=90, early_stop=False, shared_bounds=shared, timing=True)
        a = plan.project(target, r, **kw)
        assert plan.last_timing()["resident"] == 1
        s = plan.project(target, r, streaming=True, **kw)
        assert rel_err(to_np(a.y), to_np(s.y)) <= bar / 10
        assert rel_err(to_np(a.multipliers), to_np(s.multipliers)) <= bar
        kw = dict(max_iterations=600, tolerance=2e-2, shared_bounds=shared)
        a = plan.project(target, r, **kw)
        s = plan.project(target, r, streaming=True, **kw)
        ia, is_ = to_np(a.iterations), to_np(s.iterations)
        same = ia == is_
        assert same.all() if dtype == np.float64 else same.mean() >= 0.9
        if 2 * (me + mi) < n:
            assert (ia < 600).any()  # some samples stop, at their own iterations
        assert rel_err(to_np(a.y)[same], to_np(s.y)[same]) <= bar
        assert rel_err(to_np(a.multipliers)[same], to_np(s.multipliers)[same]) <= bar
        np.testing.assert_array_equal(to_np(a.status)[same], to_np(s.status)[same])


@pytest.mark.parametrize("waves", [1, 2, 3, 7, 9, 10, 11, 12, 13, 14, 15])
def test_stop_test_wavefront_sums_every_wavefront(waves):
    """The stop test's wavefront adds the others' terms in groups of eight, four, two and
    one: counts as on the streaming passes for every remainder."""
    require_gpu()
    B, n = 4, 64 * waves - 1
    w = workloads.ragged_rows(90 + waves, n=n, me=n // 20 + 1, mi=n // 8 + 1, wmin=2, wmax=5,
                              batch=B)
    plan = plan_for(canonical_from_workload(w), dtype=np.float64)
    rhs = np.tile(w.rhs, (B, 1))
    kw = dict(max_iterations=600, tolerance=1e-2)
    a = plan.project(w.target, rhs, **kw)
    s = plan.project(w.target, rhs, streaming=True, **kw)
    np.testing.assert_array_equal(to_np(a.iterations), to_np(s.iterations))
    np.testing.assert_array_equal(to_np(a.status), to_np(s.status))
    assert rel_err(to_np(a.y), to_np(s.y)) <= 1e-10


@pytest.mark.parametrize("iters", [1, 2, 3])
def test_solo_short_runs(iters):
    """The stop test trails the loop: runs that end before its first verdicts, and samples
    accepted at their first iterations (targets inside the polyhedron)."""
    require_gpu()
    B, n = 6, 70
    w = workloads.ragged_rows(9, n=n, me=0, mi=12, wmin=2, wmax=5, batch=B)
    canon = canonical_from_workload(w)
    plan = plan_for(canon, dtype=np.float64)
    rhs = np.tile(w.rhs, (B, 1))
    target = w.target.copy()
    target[::2] = 1e-3 * target[::2]  # feasible (the rows allow the origin's neighbourhood)
    rhs[:, :12] = np.abs(rhs[:, :12]) + 1.0
    kw = dict(max_iterations=iters, tolerance=1e-6)
    a = plan.project(target, rhs, **kw)
    s = plan.project(target, rhs, streaming=True, **kw)
    np.testing.assert_array_equal(to_np(a.iterations), to_np(s.iterations))
    np.testing.assert_array_equal(to_np(a.status), to_np(s.status))
    assert (to_np(a.status)[::2] == 0).all()
    assert rel_err(to_np(a.y), to_np(s.y)) <= 1e-12


@pytest.mark.parametrize("n,me,mi,B", [(70, 12, 30, 9), (300, 40, 90, 5), (1000, 80, 200, 3)])
@pytest.mark.parametrize("early", [False, True])
def test_solo_values_and_qp_match_streaming(n, me, mi, B, early):
    """Per-sample coefficients and the diagonal QP (shared and per-sample coefficients)."""
    require_gpu()
    rng = np.random.default_rng(n)
    w = workloads.ragged_rows(300 + n, n=n, me=me, mi=mi, wmin=2, wmax=10, batch=B)
    canon = canonical_from_workload(w)
    m = me + mi
    values = np.tile(w.data, (B, 1))
    general = w.indptr[m]
    values[:, :general] *= rng.uniform(0.8, 1.2, (B, general))
    rhs = np.tile(w.rhs, (B, 1))
    kw = dict(max_iterations=400, tolerance=1e-3, early_stop=early)
    for accelerated in (False, True):
        plan = plan_for(canon, dtype=np.float64, accelerated=accelerated)
        a = plan.project(w.target, rhs, values=values, **kw)
        s = plan.project(w.target, rhs, values=values, streaming=True, **kw)
        np.testing.assert_array_equal(to_np(a.iterations), to_np(s.iterations))
        assert rel_err(to_np(a.y), to_np(s.y)) <= 1e-10
        assert rel_err(to_np(a.multipliers), to_np(s.multipliers)) <= 1e-10
        rows = type(canon)(n=n, me=me, rows=canon.rows[:m], coef=canon.coef[:m])
        plan = plan_for(rows, dtype=np.float64, accelerated=accelerated, bound_presolve=False)
        q, c = rng.uniform(0.5, 2.0, (B, n)), rng.normal(0.0, 1.5, (B, n))
        lo, hi = np.full((B, n), -1.0), np.full((B, n), 1.0)
        y0 = 0.1 * rng.normal(size=(B, n))
        for v in (None, values[:, :general]):
            a = plan.qp_solve(q, c, rhs[:, :m], lo, hi, values=v, y0=y0, **kw)
            s = plan.qp_solve(q, c, rhs[:, :m], lo, hi, values=v, y0=y0, streaming=True, **kw)
            np.testing.assert_array_equal(to_np(a.iterations), to_np(s.iterations))
            assert rel_err(to_np(a.y), to_np(s.y)) <= 1e-10
            assert rel_err(to_np(a.multipliers), to_np(s.multipliers)) <= 1e-10


@pytest.mark.parametrize("n,me,mi,wmax,B", [
    (70, 12, 30, 41, 5),     # the wavefront of the stop test beside two of rows and columns
    (250, 20, 40, 43, 515),  # four wavefronts without it
])
def test_solo_stop_test_with_long_rows(n, me, mi, wmax, B):
    """Rows whose entries past the registers take the loop of four at a time and its
    remainder, in the fp64 kernels with the stop test."""
    require_gpu()
    rng = np.random.default_rng(n)
    w = workloads.ragged_rows(500 + n, n=n, me=me, mi=mi, wmin=2, wmax=wmax, batch=B)
    canon = canonical_from_workload(w)
    m = me + mi
    rhs = np.tile(w.rhs, (B, 1))
    values = np.tile(w.data, (B, 1))
    kw = dict(max_iterations=300, tolerance=1e-2)
    plan = plan_for(canon, dtype=np.float64)
    rows = type(canon)(n=n, me=me, rows=canon.rows[:m], coef=canon.coef[:m])
    qplan = plan_for(rows, dtype=np.float64, bound_presolve=False)
    q, one = rng.uniform(0.5, 2.0, (B, n)), np.ones((B, n))
    for call in (lambda **k: plan.project(w.target, rhs, **k, **kw),
                 lambda **k: plan.project(w.target, rhs, values=values, **k, **kw),
                 lambda **k: qplan.qp_solve(q, -w.target, rhs[:, :m], -one, one, **k, **kw)):
        a, s = call(), call(streaming=True)
        np.testing.assert_array_equal(to_np(a.iterations), to_np(s.iterations))
        assert rel_err(to_np(a.y), to_np(s.y)) <= 1e-10
        assert rel_err(to_np(a.multipliers), to_np(s.multipliers)) <= 1e-10


@pytest.mark.parametrize("n,me,mi,B,dtype", [
    (4097, 60, 200, 3, np.float64),     # just beyond the tile kernels
    (4200, 500, 3596, 2, np.float64),   # 4096 rows: K y+ in registers, both loops
    (4200, 500, 3597, 2, np.float64),   # 4097: K y+ in LDS; fixed iterations on the passes
    (15000, 100, 300, 2, np.float64),
    (9000, 700, 1500, 66, np.float32),
    (30000, 500, 1500, 2, np.float32),
])
def test_solo_wide_matches_streaming(n, me, mi, B, dtype):
    """Several rows and columns per thread (k_solo_wide), against the streaming passes."""
    require_gpu()
    w = workloads.ragged_rows(800, n=n, me=me, mi=mi, wmin=2, wmax=9, batch=B)
    from purin_amd.plan import Plan

    rhs = np.tile(w.rhs, (B, 1)).astype(dtype)
    target = w.target.astype(dtype)
    bar = TOL[dtype]
    scaled = rhs.copy()
    scaled[:, me + mi:] *= np.linspace(0.8, 1.2, B).astype(dtype)[:, None]
    for accelerated in (False, True):
        plan = Plan(n, me, w.rows_total - me, w.indptr, w.indices, w.data, dtype=dtype,
                    accelerated=accelerated)
        for r, shared in ((rhs, True), (scaled, False)):
            kw = dict(max_iterations=80, early_stop=False, shared_bounds=shared, timing=True)
            a = plan.project(target, r, **kw)
            assert plan.last_timing()["resident"] == (1 if me + mi <= 4096 else 0)
            s = plan.project(target, r, streaming=True, **kw)
            assert rel_err(to_np(a.y), to_np(s.y)) <= bar / 10
            assert rel_err(to_np(a.multipliers), to_np(s.multipliers)) <= bar
            kw = dict(max_iterations=400, tolerance=5e-2, shared_bounds=shared, timing=True)
            a = plan.project(target, r, **kw)
            assert plan.last_timing()["resident"] == 1
            s = plan.project(target, r, streaming=True, **kw)
            same = to_np(a.iterations) == to_np(s.iterations)
            assert same.all() if dtype == np.float64 else same.mean() >= 0.9
            assert rel_err(to_np(a.y)[same], to_np(s.y)[same]) <= bar
            assert rel_err(to_np(a.multipliers)[same], to_np(s.multipliers)[same]) <= bar


@pytest.mark.parametrize("n,me,mi,few,many,dtype", [
    (24, 4, 9, 1, 16384, np.float64), (1021, 61, 120, 3, 1025, np.float64),
    (1024, 0, 2, 2, 1025, np.float64), (333, 1, 0, 2, 6144, np.float32)])
def test_final_passes_one_column_per_wavefront(n, me, mi, few, many, dtype):
    """The final diagnostics and the multiplier recovery take one row and column per
    wavefront in small batches of small problems and eight otherwise: a few samples alone
    give what they give within a batch beyond the rule's line."""
    require_gpu()
    w = workloads.ragged_rows(50 + n, n=n, me=me, mi=mi, wmin=2, wmax=4, batch=many)
    plan = plan_for(canonical_from_workload(w), dtype=dtype, accelerated=False)
    rhs = np.tile(w.rhs, (many, 1)).astype(dtype)
    target = w.target.astype(dtype)
    kw = dict(shared_bounds=False, max_iterations=40, early_stop=False)
    a = plan.project(target, rhs, **kw)
    s = plan.project(target[:few], rhs[:few], **kw)
    bar = TOL[dtype]
    for f in ("y", "multipliers", "slacks", "residual"):
        assert rel_err(to_np(getattr(s, f)), to_np(getattr(a, f))[:few]) <= bar, f
    for f in ("status", "finite", "eligible", "iterations"):
        np.testing.assert_array_equal(to_np(getattr(s, f)), to_np(getattr(a, f))[:few])


@pytest.mark.parametrize("n,me,mi,dense", [(70, 12, 30, False), (1500, 100, 200, False),
                                           (4200, 200, 300, False), (60, 12, 25, True)])
def test_timing_counts_the_iterations_that_ran(n, me, mi, dense):
    """With the stop test the timed iterations are the longest sample's, whichever kernel ran
    them (one workgroup per sample, the tiles, several rows per thread, the dense adapter)."""
    require_gpu()
    B, limit = 6, 5000
    w = workloads.ragged_rows(17, n=n, me=me, mi=mi, wmin=2, wmax=5, batch=B)
    canon = canonical_from_workload(w)
    kw = dict(tolerance=1e-2, max_iterations=limit, timing=True)
    if dense:
        plan = plan_for(canon, dtype=np.float64, bound_presolve=False, row_scaling=False,
                        norm_bound=False)
        one = np.ones((B, n))
        rhs = np.tile(w.rhs, (B, 1))
        counts = to_np(plan.dense_solve(one, -w.target, rhs, -one, one, **kw)[2])
    else:
        plan = plan_for(canon, dtype=np.float64)
        counts = to_np(plan.project(w.target, np.tile(w.rhs, (B, 1)), **kw).iterations)
    t = plan.last_timing()
    assert t["resident"] == 1 and t["iterations"] == counts.max() < limit


def test_plan_keeps_slices_only_where_a_kernel_reads_them():
    """Two dense rows of 60,000 columns pad 62 others in the sliced rows, 60 MB; no kernel
    that reads the slices holds such vectors."""
    torch = require_gpu()
    from purin_amd.plan import Plan

    n = 60000
    ptr, idx = np.array([0, n, 2 * n]), np.tile(np.arange(n), 2)
    val = np.random.default_rng(1).normal(size=2 * n)
    Plan(8, 1, 1, np.array([0, 2, 4]), np.array([0, 1, 2, 3]), np.ones(4))  # the library's own
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    plan = Plan(n, 2, 0, ptr, idx, val)
    assert free - torch.cuda.mem_get_info()[0] < 32e6
    y = plan.project(np.zeros((1, n)), np.array([[1.0, -2.0]]), max_iterations=400).y
    np.testing.assert_allclose(to_np(y)[0] @ val.reshape(2, n).T, [1.0, -2.0], atol=1e-6)
