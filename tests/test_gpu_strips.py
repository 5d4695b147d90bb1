"""Strip sweeps at the sizes where their layout changes, against the oracle.

A strip holds 7, 10 or 14 sweep rows, its recurrences walk chunks of 8 levels
from each column's first free level, and a column's levels are dealt to groups
of 64 lanes.  The cases sit at the edges of these: sweeps one row above and
below a strip's rows, columns whose level count is not a multiple of a chunk,
columns cut off by the grid's top (a different count in every column), more
than 64 levels above the ground, and buildings that take the W sweep's columns
over one group.  Every field is compared bit for bit: the arithmetic is the
reference's, operation by operation.
"""
import numpy as np
import pytest

from gral_amd import domain
from tests.helpers import FIELDS, KE_FIELDS, diff_report


def _city(nii, njj, vcf, model=1, width=8, hmax=14.0, dz1=1.0, stretch=1.01, direction=250.0, seed=5, tower=None):
    bl = domain.city_buildings(nii, njj, 2.0, seed, density=0.2, fmin=4.0, fmax=12.0, hmin=3.0, hmax=hmax, margin=2)
    if tower:
        bl.append(domain.Building(6, 9, 5, 8, tower))
    c = domain.build_case(f"s{nii}x{njj}x{vcf}", nii, njj, bl, dx=2.0, dz1=dz1, stretch=stretch, vertcellsff=vcf, speed10=4.0,
                          direction=direction, z0=0.5, turbulence_model=model, iterations=3)
    c.simd_width = width
    return c


def _check(c, got, ref):
    fields = FIELDS + (KE_FIELDS if c.turbulence_model != 1 else ())
    for f, r in diff_report(got, ref, fields).items():
        assert r["n_bits_differ"] == 0, (c.name, f, r)
    assert got["stats"]["mass_flux"] > 0


CASES = [
    # rows of a strip: 7 in short sweeps (9, 16 and 17 interior rows), 10 from 41 rows on
    dict(nii=11, njj=18, vcf=9), dict(nii=19, njj=9, vcf=8), dict(nii=43, njj=53, vcf=11, model=2), dict(nii=54, njj=43, vcf=10, model=0),
    # chunks of 8 levels: one level more or less, both solver widths
    dict(nii=24, njj=22, vcf=15), dict(nii=22, njj=24, vcf=16, width=16), dict(nii=23, njj=21, vcf=17, model=2),
    # columns of unlike height: the grid's top cuts them off
    dict(nii=26, njj=24, vcf=16, hmax=60.0, dz1=2.0, stretch=1.2), dict(nii=24, njj=26, vcf=12, model=2, hmax=60.0, dz1=2.0, stretch=1.25),
    # 63, 64 and 65 levels above the ground: one group of 64 lanes and two
    dict(nii=12, njj=11, vcf=63), dict(nii=11, njj=12, vcf=64, model=2), dict(nii=12, njj=13, vcf=65, width=16), dict(nii=13, njj=12, vcf=66, model=0),
    # W columns over one group: 40 levels above buildings of up to 35
    dict(nii=30, njj=29, vcf=40, hmax=40.0), dict(nii=29, njj=30, vcf=40, hmax=40.0, model=2),
    # towers: W columns over two and three groups (KADVMAX 127 and 190 and one level to either side)
    dict(nii=16, njj=15, vcf=48, tower=118.0), dict(nii=15, njj=16, vcf=49, tower=118.0, model=2), dict(nii=15, njj=15, vcf=50, tower=118.0, width=16),
    dict(nii=15, njj=14, vcf=60, tower=263.0), dict(nii=14, njj=15, vcf=61, tower=263.0, model=2), dict(nii=14, njj=14, vcf=62, tower=263.0, width=16),
    dict(nii=14, njj=13, vcf=63, tower=263.0, model=0),
]


@pytest.mark.gpu
@pytest.mark.parametrize("spec", CASES, ids=lambda s: "-".join(f"{k}{v}" for k, v in s.items()))
def test_strip_edges(spec):
    from gral_amd import pf
    from oracle import pyoracle
    c = _city(**spec)
    print(f"[strips] {c.name} model {c.turbulence_model} width {c.simd_width} KADVMAX {c.kadvmax}", flush=True)
    _check(c, pf.run(c, iterations=3), pyoracle.run(c, iterations=3))


@pytest.mark.gpu
def test_many_strips():
    """More strips of ten rows than the GPU has CUs: strips of 14 rows, against plain solves."""
    from gral_amd import pf
    cases = [_city(31, 30 + q % 3, 9, direction=5.0 * q, seed=q % 7) for q in range(90)]
    got = pf.run_batch(cases, iterations=2)
    for q in range(0, 90, 11):
        ref = pf.run(cases[q], iterations=2)
        for f, r in diff_report(got[q], ref, FIELDS).items():
            assert r["n_bits_differ"] == 0, (q, f, r)


@pytest.mark.gpu
@pytest.mark.parametrize("model", [1, 2])
def test_tower_without_strip_memory(monkeypatch, model):
    """Columns over 126 levels run per-diagonal when the strips' buffers do not fit, and a batch takes no
    such columns together with lower ones."""
    from gral_amd import pf
    from oracle import pyoracle
    c = _city(16, 15, 50, tower=118.0, model=model)
    monkeypatch.setenv("GRAL_PF_DEVICE_MB", "4")
    with pf.PrognosticFlowfield(c) as s:
        s.prepare(3)
        s.iterate(3)
        assert s.timing()["launches"] > 200                   # a launch per anti-diagonal and sweep
        got = {**s.download(), "stats": s.finish()}
    monkeypatch.delenv("GRAL_PF_DEVICE_MB")
    _check(c, got, pyoracle.run(c, iterations=3))
    with pf.PrognosticFlowfield(c) as a, pf.PrognosticFlowfield(_city(16, 15, 50, model=model)) as b:
        a.prepare(3)
        b.prepare(3)
        with pytest.raises(RuntimeError):
            pf.Batch([a, b])
