"""Device memory of the strips' hand-off words: long and narrow grids need no more of it for
their size than square ones.  31 fields and the words (about 0.6 of one) fit into a budget
of 36 fields, and the sweeps run on strips with the oracle's results."""
import pytest

from gral_amd import domain
from tests.helpers import FIELDS, diff_report


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
