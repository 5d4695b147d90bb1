"""Device memory of the strips' hand-off words: long and narrow grids need no more of it for
their size than square ones.  31 fields and the words (about 0.6 of one) fit into a budget
of 36 fields, and the sweeps run on strips with the oracle's results.  Where the words alone
find no memory the situation runs per-diagonal, with the same results; it takes its place
in a batch of situations on strips."""
import pytest

from gral_amd import domain
from tests.helpers import FIELDS, KE_FIELDS, diff_report


@pytest.mark.gpu
@pytest.mark.parametrize("nii,njj", [(700, 9), (9, 700), (300, 20)])
def test_narrow_grids(monkeypatch, nii, njj):
    from gral_amd import pf
    from oracle import pyoracle
    bl = domain.city_buildings(nii, njj, 2.0, 3, density=0.2, fmin=4.0, fmax=8.0, hmin=3.0, hmax=14.0, margin=2)
    c = domain.build_case("nb", nii, njj, bl, dx=2.0, vertcellsff=20, speed10=4.0, direction=250.0, z0=0.5, iterations=4)
    nkp = (c.kadvmax + 2 + 15) // 16 * 16
    mb = int(36 * (nii + 2) * (njj + 2) * nkp * 4 / 2**20) + 1
    monkeypatch.setenv("GRAL_PF_DEVICE_MB", str(mb))
    print(f"[budget] {nii}x{njj}, {nkp} levels, {mb} MB", flush=True)
    with pf.PrognosticFlowfield(c) as s:
        s.prepare(4)
        s.iterate(4)
        assert s.timing()["launches"] < 100
        got = s.download()
    for f, r in diff_report(got, pyoracle.run(c, iterations=4), FIELDS).items():
        assert r["n_bits_differ"] == 0, (f, r)


@pytest.mark.gpu
@pytest.mark.parametrize("model", [1, 2])
def test_words_without_memory(monkeypatch, model):
    from gral_amd import pf
    bl = domain.city_buildings(120, 110, 2.0, 3, density=0.2, fmin=4.0, fmax=12.0, hmin=3.0, hmax=14.0, margin=2)
    c = domain.build_case("wm", 120, 110, bl, dx=2.0, vertcellsff=40, speed10=4.0, direction=250.0, z0=0.5, turbulence_model=model,
                          iterations=4)
    fields = FIELDS + (KE_FIELDS if model != 1 else ())
    nkp = (c.kadvmax + 2 + 15) // 16 * 16
    field = (c.nii + 2) * (c.njj + 2) * nkp * 4 / 2**20                # 3.3 MB: the words take 2 MB
    need = (31 if model == 1 else 36) * field                          # and the columns' tables about 1 MB
    with pf.PrognosticFlowfield(c) as s:
        s.prepare(4)
        s.iterate(4)
        ref = s.download()
    seen = []
    for mb in range(int(need) - 1, int(need) + 6):
        monkeypatch.setenv("GRAL_PF_DEVICE_MB", str(mb))
        s = pf.PrognosticFlowfield(c)
        monkeypatch.delenv("GRAL_PF_DEVICE_MB")
        print(f"[budget] model {model}, {need:.1f} MB needed, {mb} MB", flush=True)
        with s:
            try:
                s.prepare(5)
            except RuntimeError:
                seen.append("refused")
                continue
            both = []
            if "diag" not in seen:                                     # the first that is prepared
                with pf.PrognosticFlowfield(c) as o:
                    o.prepare(4)
                    with pf.Batch([o, s]) as b:
                        b.iterate(4)
                    both = [o.download()]
            else:
                s.iterate(4)
            both.append(s.download())
            s.iterate(1)
            seen.append("strips" if s.timing()["launches"] < 50 else "diag")
            for got in both:
                for f, r in diff_report(got, ref, fields).items():
                    assert r["n_bits_differ"] == 0, (mb, f, r)
    assert sorted(set(seen), key=seen.index) == ["refused", "diag", "strips"], seen
