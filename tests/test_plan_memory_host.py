"""Device memory that a plan initialises is ready when the call returns.

A plan may be used at once on any stream, also on one that does not wait for the null stream.  The
library runs against stand-ins of the runtime's memory functions that carry out fills and copies only
when they are waited for, as the runtime may: none may be pending after the call.
"""

import subprocess
import sys
from pathlib import Path

STANDIN = r"""
#include <cstdlib>
#include <cstring>
#include <vector>
namespace {
struct Work { void* to; std::vector<char> bytes; };
std::vector<Work> queue;
}
extern "C" {
int hipMalloc(void** p, size_t n) { *p = std::malloc(n ? n : 1); std::memset(*p, 0x5a, n); return 0; }
int hipFree(void* p) { std::free(p); return 0; }
int hipMemset(void* p, int v, size_t n) { queue.push_back({p, std::vector<char>(n, char(v))}); return 0; }
int hipMemcpy(void* to, const void* from, size_t n, int) {
  queue.push_back({to, std::vector<char>((const char*)from, (const char*)from + n)});
  return 0;
}
int hipStreamSynchronize(void*) {
  for (Work& w : queue) std::memcpy(w.to, w.bytes.data(), w.bytes.size());
  queue.clear();
  return 0;
}
int hipDeviceSynchronize() { return hipStreamSynchronize(nullptr); }
int pending() { return int(queue.size()); }
}
"""

PROGRAM = r"""
import ctypes as C, sys
import numpy as np
standin = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # before the library, so that its calls go here
from fenics_nonlinear_energies_amd import native
lib = native.lib()
ptr = lambda a: a.ctypes.data
dummy = np.zeros(64)
d = native.FnePlanDesc()
d.kind, d.n_loc, d.n_geo, d.n_elem, d.n_free, d.nq, d.nnz = native.FNE_KIND_MOHR_COULOMB, 12, 5, 1, 2, 1, 4
inc_ptr, inc, pos = np.array([0, 1, 2], np.int32), np.array([0, 1], np.uint32), np.zeros(64, np.uint8)
indptr, indices = np.array([0, 2, 4], np.int32), np.array([0, 1, 0, 1], np.int32)
for name in ("edof", "egeo", "qdata", "inc_ptr", "inc", "pitem"):
    setattr(d, name, ptr(dummy))
plan = C.c_void_p()
native.check(lib.fne_plan_create(C.byref(d), C.byref(plan)), "fne_plan_create")
print("after fne_plan_create", standin.pending())
arg = lambda a, t: a.ctypes.data_as(C.POINTER(t))
native.check(lib.fne_plan_build_row_units(plan, arg(inc_ptr, C.c_int32), arg(inc, C.c_uint32), arg(pos, C.c_uint8),
                                          arg(indptr, C.c_int32), arg(indices, C.c_int32)), "row units")
print("after fne_plan_build_row_units", standin.pending())
native.check(lib.fne_plan_destroy(plan), "fne_plan_destroy")
"""


def test_fills_and_copies_of_a_new_plan_are_waited_for(tmp_path):
    src, so = tmp_path / "standin.cpp", tmp_path / "libstandin.so"
    src.write_text(STANDIN)
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-o", str(so), str(src)], check=True)
    res = subprocess.run([sys.executable, "-c", PROGRAM, str(so)], capture_output=True, text=True,
                         cwd=Path(__file__).resolve().parents[1], timeout=300)
    assert res.returncode == 0, res.stderr
    assert res.stdout.splitlines()[-2:] == ["after fne_plan_create 0", "after fne_plan_build_row_units 0"]
