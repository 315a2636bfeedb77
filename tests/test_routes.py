"""Host rules of the library, on plans made up here (CPU only): workspace sizes.

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
