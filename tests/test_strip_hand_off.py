"""Which levels one strip of a momentum sweep hands to the next (pf_strip.h).

Column a of a strip's last row reads the old values of column a in the next strip's
row 0 at all its source levels, and row 0 stores new ones over them: wherever the
read and the stored levels overlap, row 0 has to wait for a word of that column.
The header is compiled by the host compiler with the function attributes defined
away; the columns are all combinations of ground, upstream wall and top over a
small range, and those of a generated city.
"""
import ctypes
import itertools
import os
import subprocess

import numpy as np
import pytest

from gral_amd import domain

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gral_amd", "csrc")
SOURCE = r"""
#include "pf_strip.h"
template <int C> static void ranges(const int *c, const int *p, int *out) {
    const StripCol a = strip_col<C>(c[0], c[1], c[2], c[3]), b = strip_col<C>(p[0], p[1], p[2], p[3]);
    const StripLevels sent = hand_sent<C>(b), need = hand_needed<C>(a, b);
    const int o[10] = {strip_first<C>(a), a.kend, a.VI, strip_first<C>(b), b.kend, b.VI, sent.lo, sent.hi, need.lo, need.hi};
    for (int q = 0; q < 10; ++q) out[q] = o[q];
}
extern "C" void ranges_all(int comp, int n, const int *c, const int *p, int *out) {
    for (int q = 0; q < n; ++q)
        (comp == 0 ? ranges<0> : comp == 1 ? ranges<1> : ranges<2>)(c + 4 * q, p + 4 * q, out + 10 * q);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("strip")
    src, out = os.path.join(str(d), "r.cpp"), os.path.join(str(d), "r.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__host__=", "-D__device__=", "-D__forceinline__=inline",
                    "-I", CSRC, "-o", out, src], check=True)
    return ctypes.CDLL(out)


def _ranges(lib, comp, c, p):
    c, p = (np.ascontiguousarray(x, dtype=np.int32) for x in (c, p))
    out = np.zeros((len(c), 10), dtype=np.int32)
    ip = ctypes.POINTER(ctypes.c_int)
    lib.ranges_all(comp, len(c), *(x.ctypes.data_as(ip) for x in (c, p, out)))
    return out.T


def _check(lib, comp, c, p):
    """c: columns of a row 0, p: their neighbours in the strip before; returns how many pairs update no common
    level although p reads levels that c stores."""
    cs, ce, cv, ps, pe, pv, sl, sh, nl, nh = _ranges(lib, comp, c, p)
    on = (cv >= 0) & (pv >= 0)
    waits = nl <= nh
    clash = on & (np.maximum(ce, ps) <= np.minimum(cv, pv))          # p reads old levels that c stores
    assert not (clash & ~waits).any()
    assert not (waits & ~on).any()
    # every awaited word is sent, and every new value of p at a source level of c is awaited
    assert ((nl >= sl) & (nh <= sh))[on & waits].all()
    new = on & (np.maximum(cs, pe) <= np.minimum(cv, pv))
    assert ((nl <= np.maximum(cs, pe)) & (nh >= np.minimum(cv, pv)))[new].all()
    return int((clash & ~new).sum())


@pytest.mark.parametrize("comp", [0, 1, 2])
def test_every_clash_has_a_wait(lib, comp):
    cols = [(0, -1, 0, 0), (3, 9, 0, 3 | 3 << 16)]                   # outside the sub-domains
    vcf = 8
    for kk, wall, cut, nkk in itertools.product((0, 1, 2, 5, 6, 7, 8, 9, 16, 20), (0, 3, 6, 7, 8, 9, 13, 30), (0, 1), (200, 12)):
        vi = min(nkk - 1, kk + vcf)
        if vi > kk:
            m = max(kk, wall)
            cols.append((kk, vi, (kk + 1 if cut == 0 else 1) | 1 << 16, m | m << 16))
    pairs = list(itertools.product(cols, cols))
    n = _check(lib, comp, [a for a, _ in pairs], [b for _, b in pairs])
    assert (n > 0) == (comp != 2)                                    # the layouts in question are among them


@pytest.mark.parametrize("nii,njj,layers,city", [(200, 190, 16, 2), (237, 205, 20, 11)])
def test_cities(lib, nii, njj, layers, city):
    """Generated cities hold such columns; both directions of the rows, every row as a strip's last one."""
    c = domain.build_case("h", nii, njj, domain.city_buildings(nii, njj, 2.0, city), dx=2.0, vertcellsff=layers, direction=235.0,
                          iterations=4)
    kk = c.kkart.astype(np.int32)
    kmi, kmj = kk.copy(), kk.copy()
    kmi[1:] = np.maximum(kk[1:], kk[:-1])
    kmj[:, 1:] = np.maximum(kk[:, 1:], kk[:, :-1])
    meta = np.stack([kk, np.minimum(c.nkk - 1, kk + layers), np.where(c.cutk == 0, kk + 1, 1) | (c.advdom.astype(np.int32) << 16),
                     kmi | (kmj << 16)], axis=-1)[2:nii, 2:njj]
    found = 0
    for comp, js in itertools.product((0, 1), (1, -1)):
        rows = meta[:, ::js]
        found += _check(lib, comp, rows[:, 1:].reshape(-1, 4), rows[:, :-1].reshape(-1, 4))
    assert found > 0
