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
