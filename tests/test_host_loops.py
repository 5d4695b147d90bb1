"""Host loops of the C ABI (pf_host.h), compiled by the host compiler.

The particles' cells are checked in blocks on the host threads: the first one outside the
grid is found at the blocks' edges, and for as many particles as the argument's type holds.
A loop that cannot start its threads runs their parts itself, each once."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gral_amd", "csrc")
SOURCE = r"""
#include "pf_host.h"
extern "C" int32_t outside(int32_t n, const int32_t *i, const int32_t *j, int nii, int njj) { return first_outside(n, i, j, nii, njj); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("host")
    src, out = os.path.join(str(d), "h.cpp"), os.path.join(str(d), "h.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-fPIC", "-shared", "-I", CSRC, "-o", out, src], check=True)
    return ctypes.CDLL(out)


def _outside(lib, ci, cj, n=None, nii=7, njj=9):
    ip = ctypes.POINTER(ctypes.c_int32)
    return lib.outside(len(ci) if n is None else n, ci.ctypes.data_as(ip), cj.ctypes.data_as(ip), nii, njj)


@pytest.mark.parametrize("n", [0, 1, 65535, 65536, 65537, 200001])
def test_first_particle_outside(lib, n):
    ci, cj = np.full(n, 7, np.int32), np.full(n, 9, np.int32)
    assert _outside(lib, ci, cj) == n
    for p in sorted({0, n // 2, 65535, 65536, n - 1}):
        if 0 <= p < n:
            for a, v in ((ci, 8), (ci, 0), (cj, 10), (cj, 0)):
                old, a[p], a[-1] = int(a[p]), v, -5
                assert _outside(lib, ci, cj) == p
                a[-1] = old
                a[p] = old


@pytest.mark.parametrize("n", [2**31 - 65536, 2**31 - 65535, 2**31 - 1])
def test_largest_counts(lib, n):
    z = np.zeros(n, np.int32)                             # cells 0: outside; pages of zeros that are only read take no memory
    assert _outside(lib, z, z, n) == 0


THREADS = r"""
#include <cassert>
#include <cerrno>
#include <cstdio>
#include <dlfcn.h>
#include <pthread.h>
#include "pf_host.h"
static int left;
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *x) {
    typedef int (*Fn)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    if (left-- <= 0) return EAGAIN;
    return ((Fn)dlsym(RTLD_NEXT, "pthread_create"))(t, a, f, x);
}
int main() {
    for (int avail : {0, 1, 3, 100})
        for (long n : {1L, 2L, 15L, 16L, 17L, 1000L}) {
            left = avail;
            std::vector<std::atomic<int>> seen(n + 5);
            std::vector<std::atomic<int>> part(64);
            par_for(5, n + 5, [&](int t, long a, long b) {
                part[t]++;
                for (long k = a; k < b; ++k) seen[k]++;
            });
            for (long k = 0; k < n + 5; ++k) if (seen[k] != (k >= 5)) return 1;
            for (auto &p : part) if (p > 1) return 2;
        }
    std::puts("ok");
}
"""


def test_without_threads(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(THREADS)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", CSRC, "-o", str(exe), str(src), "-ldl"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert (r.returncode, r.stdout) == (0, "ok\n"), r.stderr
