"""Sweeps of two first-order recurrences on strips, at the edges of their layout.

The diagnostic pressure sweep: one, two and four groups of 64 levels a column,
columns too tall for the strips, strips of 7 and 10 rows that end in a partial
strip, cell sizes that are no power of two; every field bit for bit against the
oracle.  One momentum sweep: on strips bit for bit what it is with one launch
per anti-diagonal.  Its transpose: against central differences, for columns of
one and two groups of levels.  The transposed pressure sweep: against the oracle
in float64.
"""
import numpy as np
import pytest

from gral_amd import domain
from tests.test_gpu_diagnostic import FIELDS, _compare

DIAG = [
    # nii, njj, dx, first level, stretch: NKK 25, 62, 63, 126, 127, 221, 254 and 255
    (9, 8, 2.0, 2.0, 1.2), (16, 17, 3.0, 1.0, 1.067), (43, 42, 2.0, 1.0, 1.0655), (17, 45, 2.0, 1.0, 1.02425),
    (44, 9, 2.5, 1.0, 1.02395), (12, 11, 2.0, 1.0, 1.01), (10, 12, 2.0, 1.0, 1.00785), (11, 10, 2.0, 1.0, 1.0078),
]


@pytest.mark.gpu
@pytest.mark.parametrize("nii,njj,dx,dz1,stretch", DIAG)
def test_diagnostic_edges(nii, njj, dx, dz1, stretch):
    bl = domain.city_buildings(nii, njj, dx, 3, density=0.25, fmin=3.0, fmax=9.0, hmin=3.0, hmax=25.0, margin=1)
    c = domain.build_case("dgs", nii, njj, bl, dx=dx, dz1=dz1, stretch=stretch, vertcellsff=8, direction=215.0, iterations=2)
    _compare(c, 0, 2)


@pytest.mark.gpu
@pytest.mark.parametrize("width", [8, 16])
@pytest.mark.parametrize("nii,njj", [(9, 11), (18, 16), (46, 43)])
def test_momentum_sweep_kinds(monkeypatch, nii, njj, width):
    from gral_amd import pf
    bl = domain.city_buildings(nii, njj, 2.0, 5, density=0.2, fmin=4.0, fmax=12.0, hmin=3.0, hmax=14.0, margin=2)
    c = domain.build_case("ms", nii, njj, bl, dx=2.0, vertcellsff=17, direction=235.0, z0=0.5, iterations=4)
    c.simd_width = width
    out = {}
    for sw in ("strip", "diag"):
        monkeypatch.setenv("GRAL_PF_SWEEP", sw)
        with pf.PrognosticFlowfield(c) as s:
            s.prepare(iterations=4)
            s.iterate(3)
            for comp in range(3):
                print(f"[line strips] sweep {comp} of {nii}x{njj} {sw}", flush=True)
                s.momentum_sweep(comp)
            out[sw] = s.download()
    for f in FIELDS:
        assert np.array_equal(out["strip"][f].view(np.uint32), out["diag"][f].view(np.uint32)), f


@pytest.mark.gpu
@pytest.mark.parametrize("comp", [0, 1, 2])
@pytest.mark.parametrize("nii,njj,vcf,width", [(9, 11, 17, 8), (46, 43, 17, 16), (12, 45, 70, 8), (43, 12, 60, 16)])
def test_momentum_vjp_edges(nii, njj, vcf, width, comp):
    # <g, M(x + h d) - M(x - h d)> / 2h against <VJP(g), d>: for random g and d over N
    # cells both are sums of N terms of random sign, of size sqrt(N) where the
    # Jacobian is near the identity; the differences' float rounding (6e-8 / 2h with
    # h = 1e-3) leaves 3e-5 of that, the bound is 1e-3 of it
    from gral_amd import pf
    f = ("uk", "vk", "wk")[comp]
    bl = domain.city_buildings(nii, njj, 2.0, 5, density=0.2, fmin=4.0, fmax=12.0, hmin=3.0, hmax=14.0, margin=2)
    c = domain.build_case("mv", nii, njj, bl, dx=2.0, vertcellsff=vcf, direction=235.0, z0=0.5, iterations=6)
    c.simd_width, c.relax = width, 1.0
    lev = np.zeros(c.uk.shape, dtype=bool)
    lev[:, :, :c.kadvmax + 2] = True
    rng = np.random.default_rng(7 + comp)
    g = np.where(lev, rng.standard_normal(c.uk.shape), 0.0).astype(np.float32)
    d = np.where(lev, rng.standard_normal(c.uk.shape), 0.0)
    print(f"[line strips] vjp of {f}, {nii}x{njj}, {c.kadvmax + 2} levels, width {width}", flush=True)
    with pf.PrognosticFlowfield(c) as s:
        s.prepare(iterations=6)
        s.iterate(2)
        base = {k: v.copy() for k, v in s.download().items() if k in ("uk", "vk", "wk")}
        s.momentum_sweep(comp)
        ad = s.momentum_vjp(g)
        s.restore_ckpt()
        h = 1e-3 * float(np.abs(base[f][lev]).max())
        x, y = [], []
        for sgn in (1.0, -1.0):
            v = {k: a.copy() for k, a in base.items()}
            v[f] = (base[f].astype(np.float64) + sgn * h * d).astype(np.float32)
            s.set_velocity(v["uk"], v["vk"], v["wk"])
            s.momentum_sweep(comp)
            x.append(v[f].astype(np.float64))
            y.append(s.download()[f].astype(np.float64))
    fd = float((g * (y[0] - y[1])).sum()) / (2 * h)
    av = float((ad.astype(np.float64) * (x[0] - x[1])).sum()) / (2 * h)
    assert abs(av - fd) <= 1e-3 * np.sqrt(lev.sum()), (av, fd)


VJP = [
    # one, two and four groups of 64 levels; strips of 7 and 10 rows; columns cut off by the grid's top, whose
    # eliminations start from an earlier column's value; columns per anti-diagonal
    dict(nii=9, njj=11, vcf=9), dict(nii=46, njj=43, vcf=17, hmax=30.0), dict(nii=12, njj=45, vcf=70),
    dict(nii=14, njj=13, vcf=63, tower=263.0), dict(nii=26, njj=24, vcf=16, hmax=60.0, dz1=2.0, stretch=1.2),
    dict(nii=24, njj=60, vcf=12, hmax=60.0, dz1=2.0, stretch=1.25), dict(nii=18, njj=16, vcf=8, sweep="diag"),
]


@pytest.mark.gpu
@pytest.mark.parametrize("spec", VJP, ids=lambda s: "-".join(f"{k}{v}" for k, v in s.items()))
def test_window_vjp_edges(monkeypatch, spec):
    # <g, F(x + d) - F(x)> by the oracle in float64 against <VJP(g), d>: both of size
    # sqrt(N) for random g and d over N cells; float32 rounding over the window's
    # sweeps (6e-8 times some hundred operations) is below the bound of 1e-4 of that
    from gral_amd import pf
    from oracle import pyoracle
    from tests.test_gpu_adjoint import _direction, _dot, _shifted
    spec = dict(spec)
    monkeypatch.setenv("GRAL_PF_SWEEP", spec.pop("sweep", "strip"))
    vcf, hmax, tower = spec.pop("vcf"), spec.pop("hmax", 14.0), spec.pop("tower", None)
    bl = domain.city_buildings(spec["nii"], spec["njj"], 2.0, 5, density=0.2, fmin=4.0, fmax=12.0, hmin=3.0, hmax=hmax, margin=2)
    if tower:
        bl.append(domain.Building(6, 9, 5, 8, tower))
    c = domain.build_case("wv", buildings=bl, dx=2.0, vertcellsff=vcf, direction=235.0, z0=0.5, iterations=4, **spec)
    lev = np.zeros(c.uk.shape, dtype=bool)
    lev[:, :, :c.kadvmax + 2] = True
    rng = np.random.default_rng(3)
    g = tuple(np.where(lev, rng.standard_normal(c.uk.shape), 0.0).astype(np.float32) for _ in range(3))
    print(f"[line strips] window vjp {c.nii}x{c.njj}, {c.kadvmax + 2} levels", flush=True)
    with pf.PrognosticFlowfield(c) as s:
        s.prepare(iterations=4)
        s.forward_ckpt(4)
        v = s.vjp(*g)
    d = _direction(c, 11)
    base = pyoracle.run(c, iterations=4, project=0, fp64=True)
    pert = pyoracle.run(_shifted(c, d, 1.0), iterations=4, project=0, fp64=True)
    lhs = _dot(g, [pert[f] - base[f] for f in ("uk", "vk", "wk")])
    assert abs(_dot(v, d) - lhs) <= 1e-4 * np.sqrt(3.0 * lev.sum()), (_dot(v, d), lhs)
