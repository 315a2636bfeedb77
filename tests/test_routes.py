"""Host rules of the library, on plans made up here (CPU only): workspace sizes and which
kernel runs a call.

The rules read a plan's sizes and row and column widths alone, so a plan whose device arrays
are empty serves.  A few lines of C++ against the library's own headers make one.
"""

import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from purin_amd import build as B

HARNESS = r"""
#include <algorithm>
#include "forward.hpp"
#include "gmres.hpp"
#include "solo.hpp"

using namespace purin;

// m kept rows and n columns of the given widths, M rows in all
extern "C" purin_cp_plan* route_plan(int f64, int64_t n, int64_t m, int64_t M, const int32_t* rw,
                                     const int32_t* cw) {
  auto* p = new purin_cp_plan;
  p->dtype = f64 ? PURIN_CP_F64 : PURIN_CP_F32;
  p->n = n;
  p->m = m;
  p->M = M;
  p->mi = M;
  p->sl_ok = n < 65535 && m < 65535;
  auto slices = [](const int32_t* w, int64_t count, std::vector<int32_t>& wide, int64_t& total) {
    std::vector<int32_t> d(w, w + count);
    std::sort(d.rbegin(), d.rend());
    for (int64_t s = 0; s < count; s += 64) {
      wide.push_back(d[s]);
      total += 64 * (int64_t)d[s];
    }
    return (int32_t)wide.size();
  };
  p->sl_nsr = slices(rw, m, p->sl_rw, p->sl_rn);
  p->sl_nsc = slices(cw, n, p->sl_cw, p->sl_cn);
  for (int64_t i = 0; i < m; ++i) p->nnz += rw[i];
  p->nnz_full = p->nnz + M - m;
  p->bound.assign((size_t)(M - m), 0);
  return p;
}
extern "C" void route_free(purin_cp_plan* p) { delete p; }
extern "C" int route_solo(const purin_cp_plan* p, int64_t batch, int early, int values) {
  return solo_fits(p, batch, early != 0, values != 0);
}
extern "C" int route_wide(const purin_cp_plan* p, int64_t batch, int early) {
  return solo_wide_fits(p, batch, early != 0);
}
extern "C" int64_t route_gmr(const purin_cp_plan* p, int64_t restart, int dense) {
  return gmr_batch(p, restart, dense != 0);
}
extern "C" int64_t route_workspace(const purin_cp_plan* p, int entry, int64_t batch) {
  return purin_cp_workspace_bytes(p, entry, batch, nullptr);
}
"""


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    d = tmp_path_factory.mktemp("routes")
    src, out = d / "routes.hip", d / "libroutes.so"
    src.write_text(HARNESS)
    libdir = os.path.dirname(B.LIB)
    subprocess.run([B._hipcc(), "-std=c++17", "-O1", "-fPIC", "-shared", "--offload-host-only",
                    "-x", "hip", "-I", B.CSRC, str(src), "-L", libdir,
                    "-l:" + os.path.basename(B.LIB), "-Wl,-rpath," + libdir, "-o", str(out)],
                   check=True, capture_output=True)
    lib = C.CDLL(str(out))
    i32, i64, vp = C.POINTER(C.c_int32), C.c_int64, C.c_void_p
    lib.route_plan.restype = vp
    lib.route_plan.argtypes = [C.c_int, i64, i64, i64, i32, i32]
    lib.route_free.argtypes = [vp]
    lib.route_solo.argtypes = [vp, i64, C.c_int, C.c_int]
    lib.route_wide.argtypes = [vp, i64, C.c_int]
    lib.route_gmr.restype = i64
    lib.route_gmr.argtypes = [vp, i64, C.c_int]
    lib.route_workspace.restype = i64
    lib.route_workspace.argtypes = [vp, C.c_int, i64]
    return lib


class _Plan:
    """A plan of m rows of the given widths over n columns (spread evenly), with box rows."""

    def __init__(self, lib, n, widths, dtype=np.float64, col_widths=None):
        rw = np.asarray(widths, np.int32)
        if col_widths is None:
            col_widths = np.full(n, rw.sum() // n)
            col_widths[:rw.sum() - col_widths.sum()] += 1
        cw = np.asarray(col_widths, np.int32)
        self.lib = lib
        self.p = lib.route_plan(int(dtype == np.float64), n, rw.size, rw.size + 2 * n,
                                rw.ctypes.data_as(C.POINTER(C.c_int32)),
                                cw.ctypes.data_as(C.POINTER(C.c_int32)))

    def __del__(self):
        self.lib.route_free(self.p)

    def solo(self, batch, early, values=False):
        return bool(self.lib.route_solo(self.p, batch, int(early), int(values)))

    def wide(self, batch, early):
        return bool(self.lib.route_wide(self.p, batch, int(early)))

    def gmr(self, restart, dense=False):
        return self.lib.route_gmr(self.p, restart, int(dense))

    def workspace(self, entry, batch):
        from purin_amd import _lib

        return self.lib.route_workspace(self.p, _lib.ENTRY[entry], batch)


@pytest.mark.parametrize("n,m,dtype", [(24, 13, np.float64), (60, 37, np.float64),
                                       (60, 37, np.float32), (1024, 900, np.float64),
                                       (6000, 2100, np.float64)])
@pytest.mark.parametrize("entry", ["solve", "project", "project_values", "qp_solve"])
def test_workspace_of_a_batch_serves_smaller_ones(routes, n, m, dtype, entry):
    """Callers size one workspace for the largest batch they make."""
    plan = _Plan(routes, n, np.full(m, 5), dtype)
    sizes = [plan.workspace(entry, b) for b in range(1, 70000, 61)]
    assert min(sizes) > 0
    assert all(a <= b for a, b in zip(sizes, sizes[1:]))


def _rows(n, m, w, wide=0, wide_w=0):
    return np.concatenate((np.full(wide, wide_w), np.full(m - wide, w))).astype(int)


@pytest.mark.parametrize("n,m,w,wide,dtype,early,fixed", [
    # the batches up to which one workgroup per sample pays (None: all), as measured
    (250, 75, 5, (0, 0), np.float64, None, None),
    (250, 75, 5, (0, 0), np.float32, None, None),
    (500, 150, 5, (0, 0), np.float32, None, 1024),
    (200, 21, 4, (1, 200), np.float64, 256, 256),   # one workgroup's entries fill the LDS
    (240, 21, 4, (1, 240), np.float32, 512, 256),
    (120, 21, 4, (1, 120), np.float64, None, None),  # two fit
    (300, 65, 4, (5, 150), np.float64, 256, 256),
    (300, 65, 4, (5, 150), np.float32, 1024, 512),
    (250, 75, 40, (0, 0), np.float64, None, 256),
    (250, 75, 12, (0, 0), np.float32, None, 1024),
    (500, 150, 40, (0, 0), np.float64, 256, 256),
    (500, 150, 24, (0, 0), np.float32, 1024, 512),
    (700, 210, 12, (0, 0), np.float64, None, 256),
    (700, 210, 40, (0, 0), np.float64, 256, 256),
])
def test_one_workgroup_per_sample_where_it_pays(routes, n, m, w, wide, dtype, early, fixed):
    """Long rows take LDS from the workgroups that share a CU: past the batches where the tile
    kernels are faster the calls go there.  Per-sample coefficients stay."""
    widths = _rows(n, m, w, *wide)
    # columns of a random matrix: a few stand out by up to ten entries
    cols = np.full(n, widths.sum() // n)
    if widths.max() > 8:
        cols[:3] += 6
    plan = _Plan(routes, n, widths, dtype, col_widths=cols)
    for stop, last in ((True, early), (False, fixed)):
        for batch in (1, 256, 257, 512, 513, 1024, 1025, 8192):
            assert plan.solo(batch, stop) == (last is None or batch <= last), (batch, stop)
            assert plan.solo(batch, stop, values=True)


@pytest.mark.parametrize("n,m,w,wide,dtype,early,fixed", [
    # (smallest, largest) batch of the workgroup per sample, as measured
    (8000, 2000, 4, (0, 0), np.float64, (1, None), (1, None)),
    (8000, 2000, 75, (0, 0), np.float64, (1, None), (1, None)),
    (8000, 2000, 200, (0, 0), np.float64, (1, None), (129, None)),
    (8000, 2000, 50, (0, 0), np.float32, (1, None), (1, None)),
    (8000, 2000, 100, (0, 0), np.float32, (1, None), (1, 512)),
    (12000, 4000, 10, (0, 0), np.float64, (1, None), (1, None)),
    (8000, 3000, 4, (1, 8000), np.float64, (1, 512), (1, 256)),
    (8000, 3000, 4, (4, 2000), np.float64, (1, None), (1, 512)),
    (8000, 3000, 4, (64, 500), np.float64, (1, None), (1, 512)),
    (8000, 3000, 4, (4, 100), np.float64, (1, None), (1, None)),
    (8000, 4100, 4, (0, 0), np.float64, (1, None), None),  # rows beyond one group
    (4200, 200, 4, (0, 0), np.float64, (1, None), (1, None)),  # nearly empty
    (4200, 200, 12, (0, 0), np.float32, (1, None), (1, 1024)),
])
def test_wide_loop_where_it_pays(routes, n, m, w, wide, dtype, early, fixed):
    """A workgroup streams the whole matrix: wide rows, one long chain and many rounds go to
    the passes."""
    widths = _rows(n, m, w, *wide)
    plan = _Plan(routes, n, widths, dtype)
    for stop, line in ((True, early), (False, fixed)):
        for batch in (1, 64, 128, 129, 256, 257, 512, 513, 1024, 4096):
            pays = line is not None and line[0] <= batch and (line[1] is None or batch <= line[1])
            assert plan.wide(batch, stop) == pays, (batch, stop)


ALL = 2**63 - 1


@pytest.mark.parametrize("n,m,w,wide,dtype,restart,dense,batch", [
    (60, 30, 60, (0, 0), np.float64, 5, True, 1024),  # sums over the batch through one counter
    (20000, 50, 4, (0, 0), np.float64, 5, True, 0),   # beyond the LDS
    (300, 90, 5, (0, 0), np.float64, 30, False, ALL),
    (300, 90, 5, (0, 0), np.float64, 33, False, 0),
    (300, 50, 4, (1, 300), np.float64, 30, False, ALL),  # eight wavefronts share the row
    (800, 300, 4, (2, 300), np.float64, 30, False, 1024),
    (600, 300, 4, (4, 400), np.float32, 30, False, 4096),
    (1000, 300, 4, (1, 1000), np.float64, 30, False, 1024),
    (1000, 300, 4, (1, 1000), np.float32, 30, False, 2048),
    (2000, 400, 4, (8, 600), np.float64, 30, False, ALL),  # small beside the vectors
    (8000, 2500, 4, (4, 1500), np.float64, 30, False, 512),  # but one workgroup per CU
    (8000, 2500, 4, (4, 1500), np.float32, 30, False, ALL),
    (8000, 2000, 50, (0, 0), np.float64, 30, False, ALL),
    (4000, 600, 4, (20, 2000), np.float64, 30, False, 512),
    (8000, 500, 4, (1, 8000), np.float64, 30, False, 512),
    (4000, 600, 4, (20, 2000), np.float32, 30, False, 1024),
    (8000, 500, 4, (1, 8000), np.float32, 30, False, 512),
])
def test_adjoint_workgroups_where_they_pay(routes, n, m, w, wide, dtype, restart, dense, batch):
    """The largest batch whose implicit VJP runs one workgroup per sample."""
    assert _Plan(routes, n, _rows(n, m, w, *wide), dtype).gmr(restart, dense) == batch
