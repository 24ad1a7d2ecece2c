"""Shared fixtures. GPU tests are marked ``gpu``; everything else runs on CPU."""

import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "bcm-problems_amd"))
sys.path.insert(0, os.path.join(ROOT, "oracle"))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through the C ABI on the device)")


@pytest.fixture(scope="session")
def B():
    import bcmhip

    bcmhip.lib()
    return bcmhip


@pytest.fixture(scope="session")
def O():
    import oracle

    oracle.orc()
    return oracle


@pytest.fixture(scope="session")
def ctx(B):
    return B.Context()


class SweepPlan:
    """The host side of the sync-free sweeps (csrc/device/sweep_plan.hpp, no device code), compiled for the tests."""

    SRC = """
#include "sweep_plan.hpp"
using namespace bcm;
extern "C" {
int levels(int ns, const int* ia, const int* ja, int forward, int* lev) {
  int n = 0;
  for (int q = 0; q < ns; ++q) {
    const int r = forward ? q : ns - 1 - q;
    lev[r] = 0;
    for (int j = ia[r]; j < ia[r + 1]; ++j) lev[r] = std::max(lev[r], lev[ja[j]] + 1);
    n = std::max(n, lev[r] + 1);
  }
  return n;
}
int held(int b) { return strip_held(b); }
int in_strips(int b, int bytes, long ns, long levels, long nrhs) { return sweep_in_strips(b, bytes, ns, levels, nrhs); }
double wait_seconds(long levels, long deps, long blocks, long nrhs) { return sweep_wait_seconds(levels, deps, blocks, nrhs); }
int cut(int b, int bytes, int levels, int ns, const int* ia, const int* ja, const int* lev, int forward, int* rows, int* ptr,
        int* code) {
  const Strips t = cut_strips(b, bytes, levels, {ia, ia + ns + 1}, {ja, ja + ia[ns]}, {lev, lev + ns}, forward != 0);
  if (t.count) {
    std::copy(t.rows.begin(), t.rows.end(), rows);
    std::copy(t.ptr.begin(), t.ptr.end(), ptr);
    std::copy(t.code.begin(), t.code.begin() + ia[ns], code);
  }
  return t.count;
}
}
"""

    def __init__(self, folder):
        src, so = os.path.join(folder, "plan.cpp"), os.path.join(folder, "plan.so")
        with open(src, "w") as f:
            f.write(self.SRC)
        inc = os.path.join(ROOT, "bcm-problems_amd", "csrc", "device")
        subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", inc, src, "-o", so], check=True)
        self.l = ctypes.CDLL(so)
        self.l.wait_seconds.restype = ctypes.c_double
        self.l.wait_seconds.argtypes = [ctypes.c_long] * 4
        self.l.in_strips.argtypes = [ctypes.c_int, ctypes.c_int] + [ctypes.c_long] * 3

    def levels(self, ia, ja, forward):
        """(number of levels, level of each row) of dependency lists."""
        lev = np.zeros(len(ia) - 1, np.int32)
        return self.l.levels(len(lev), _ints(ia), _ints(ja), int(forward), _ints(lev)), lev

    def cut(self, b, bytes_, ia, ja, forward):
        """(strips, rows, first positions, codes) of dependency lists ia, ja; 0 strips: none."""
        n, lev = self.levels(ia, ja, forward)
        ns = len(lev)
        rows, ptr, code = np.zeros(ns, np.int32), np.zeros(ns + 1, np.int32), np.zeros(max(len(ja), 1), np.int32)
        k = self.l.cut(b, bytes_, n, ns, _ints(ia), _ints(ja), _ints(lev), int(forward), _ints(rows), _ints(ptr), _ints(code))
        return k, rows, ptr[:k + 1], code[:len(ja)]

    def factor_strips(self, f, ns, b, bytes_, nrhs):
        """(whether both sweeps of factor f run in strips, most dependencies of a
        row, whether a strip of each has two rows of one level)."""
        deps, yes, shared = 0, True, True
        for which, forward in ((0 if f.kind == 1 else 1, True), (1, False)):
            ia, ja, _ = f.arrays(which, ns)
            rows = np.repeat(np.arange(ns), np.diff(ia))
            off = rows != ja
            r, c = (ja[off], rows[off]) if forward else (rows[off], ja[off])
            o = np.lexsort((c, r))
            dia = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=ns))]).astype(np.int32)
            dja = np.ascontiguousarray(c[o], dtype=np.int32)
            deps = max(deps, int(np.diff(dia).max()))
            n, lev = self.levels(dia, dja, forward)
            k, order, ptr, _ = self.cut(b, bytes_, dia, dja, forward)
            yes = yes and k > 0 and self.l.in_strips(b, bytes_, ns, n, nrhs)
            shared = shared and any((np.diff(lev[order[ptr[q]:ptr[q + 1]]]) == 0).any() for q in range(k))
        return bool(yes), deps, shared


def _ints(a):
    assert a.dtype == np.int32 and a.flags.c_contiguous
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int))


@pytest.fixture(scope="session")
def plan(tmp_path_factory):
    return SweepPlan(str(tmp_path_factory.mktemp("plan")))


def rel(a, b):
    a = np.asarray(a, dtype=np.float64).ravel(order="F")
    b = np.asarray(b, dtype=np.float64).ravel(order="F")
    assert a.shape == b.shape, (a.shape, b.shape)
    d = np.linalg.norm(b)
    return np.linalg.norm(a - b) / (d if d > 0 else 1.0)
