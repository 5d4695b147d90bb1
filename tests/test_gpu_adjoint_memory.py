"""The transposes where device memory is short.  A momentum sweep's transpose needs 8 fields of
column data and the hand-off words where the situation has no strips; a situation for which
they do not fit runs it with one launch per anti-diagonal, to the same gradients bit for
bit."""
import numpy as np
import pytest

from gral_amd import domain


def _case(nii, njj, vcf, width=8):
    bl = domain.city_buildings(nii, njj, 2.0, 5, density=0.2, fmin=4.0, fmax=12.0, hmin=3.0, hmax=14.0, margin=2)
    c = domain.build_case("am", nii, njj, bl, dx=2.0, vertcellsff=vcf, direction=235.0, z0=0.5, iterations=6)
    c.simd_width = width
    nkp = (c.kadvmax + 2 + 15) // 16 * 16
    return c, (nii + 2) * (njj + 2) * nkp * 4 / 2**20


def _solver(monkeypatch, c, sweep, mb=None):
    from gral_amd import pf
    monkeypatch.setenv("GRAL_PF_SWEEP", sweep)
    if mb:
        monkeypatch.setenv("GRAL_PF_DEVICE_MB", str(int(mb)))
    s = pf.PrognosticFlowfield(c)
    s.prepare(6)
    monkeypatch.delenv("GRAL_PF_DEVICE_MB", raising=False)
    monkeypatch.delenv("GRAL_PF_SWEEP")
    return s


@pytest.mark.gpu
@pytest.mark.parametrize("nii,njj,vcf,width", [(140, 131, 30, 8), (121, 150, 70, 16)])
def test_momentum_vjp_without_column_data(monkeypatch, nii, njj, vcf, width):
    c, field = _case(nii, njj, vcf, width)
    g = np.random.default_rng(3).standard_normal(c.uk.shape).astype(np.float32)
    out = []
    # strips; per-diagonal with the column data, and with 27 fields and 4 MB, so without them
    for sweep, mb in (("strip", None), ("diag", None), ("diag", 27 * field + 4)):
        print(f"[adjoint memory] momentum {nii}x{njj}, field {field:.1f} MB, {sweep} {mb}", flush=True)
        assert mb is None or mb < 35 * field
        with _solver(monkeypatch, c, sweep, mb) as s:
            s.iterate(2)
            grads = []
            for comp in range(3):
                s.momentum_sweep(comp)
                grads.append(s.momentum_vjp(g))
            out.append(grads)
    for o in out[1:]:
        for a, b in zip(out[0], o):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("spec", [dict(nii=14, njj=13, vcf=62, tower=263.0, stretch=1.003),
                                  dict(nii=13, njj=15, vcf=40, tower=290.0, stretch=1.002, hmax=40.0)],
                         ids=lambda s: f"{s['nii']}x{s['njj']}")
def test_window_vjp_above_the_strips(spec):
    # columns of more than 256 levels: the transposed pressure sweep with one launch per
    # anti-diagonal, over four steps.  The bound is test_window_vjp_edges': 1e-4 of sqrt(N)
    from gral_amd import pf
    from oracle import pyoracle
    from tests.test_gpu_adjoint import _direction, _dot, _shifted
    from tests.test_gpu_strips import _city
    c = _city(**spec)
    assert c.kadvmax + 2 > 256
    lev = np.zeros(c.uk.shape, dtype=bool)
    lev[:, :, :c.kadvmax + 2] = True
    rng = np.random.default_rng(3)
    g = tuple(np.where(lev, rng.standard_normal(c.uk.shape), 0.0).astype(np.float32) for _ in range(3))
    print(f"[adjoint memory] window {c.nii}x{c.njj}, {c.kadvmax + 2} levels", flush=True)
    with pf.PrognosticFlowfield(c) as s:
        s.prepare(iterations=4)
        s.forward_ckpt(4)
        v = s.vjp(*g)
    d = _direction(c, 11)
    base = pyoracle.run(c, iterations=4, project=0, fp64=True)
    pert = pyoracle.run(_shifted(c, d, 1.0), iterations=4, project=0, fp64=True)
    lhs = _dot(g, [pert[f] - base[f] for f in ("uk", "vk", "wk")])
    assert abs(_dot(v, d) - lhs) <= 1e-4 * np.sqrt(3.0 * lev.sum()), (_dot(v, d), lhs)


@pytest.mark.gpu
def test_window_vjp_without_words(monkeypatch):
    # the smallest budget the window runs in leaves less than 1 MB, the hand-off words take more
    c, field = _case(140, 131, 30)
    nkp = (c.kadvmax + 2 + 15) // 16 * 16
    assert 2 * 8 * (c.njj // 7 + 1) * c.nii * nkp > 1 << 20
    g = [np.random.default_rng(q).standard_normal(c.uk.shape).astype(np.float32) for q in range(3)]
    out = []
    for sweep, first in (("strip", None), ("diag", int(27 * field))):
        for mb in [None] if first is None else range(first, first + 6):
            print(f"[adjoint memory] window 140x131, field {field:.1f} MB, {sweep} {mb}", flush=True)
            with _solver(monkeypatch, c, sweep, mb) as s:
                try:
                    s.forward_ckpt(4)
                except RuntimeError:
                    continue
                out.append(s.vjp(*g))
                break
    for a, b in zip(*out):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
