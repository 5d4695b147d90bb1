"""Strips whose neighbouring rows update no common level: low roofs beside walls higher
than the sub-domain's levels in a strip's last row, open ground in the next strip's
first row (U: the wall upstream in the row, V: a wall along the row before), and a
generated city that holds such columns.  The next strip must not store over the ground
before the roof's column has read it: every field bit for bit against the oracle, over a
cycle of the four sweep directions."""
import pytest

from gral_amd import domain
from tests.helpers import FIELDS, KE_FIELDS, diff_report


def _layout(model, vcf=8, nii=30, njj=31):
    bl = []
    for j in (8, njj - 7):                                # U: the last rows of the first strips, JS = 1 and -1
        for i in range(4, 13, 2):
            bl += [domain.Building(i, i, j, j, 12.5), domain.Building(i + 1, i + 1, j, j, 6.0)]
    bl += [domain.Building(16, 27, 8, 8, 12.5), domain.Building(16, 27, 9, 9, 6.0)]      # V, JS = 1
    c = domain.build_case(f"hand{model}", nii, njj, bl, dx=2.0, vertcellsff=vcf, speed10=4.0, direction=250.0, z0=0.5,
                          turbulence_model=model, iterations=4)
    kk = c.kkart.astype(int)
    assert kk[5, 8] < kk[4, 8] and kk[4, 8] >= vcf and kk[4, 8] < kk[5, 8] + vcf and kk[5, 9] == 0      # kend above the ground's levels
    assert kk[16, 9] < kk[16, 8] < kk[16, 9] + vcf and kk[16, 8] >= vcf and kk[16, 10] == 0
    return c


def _check(c):
    from gral_amd import pf
    from oracle import pyoracle
    fields = FIELDS + (KE_FIELDS if c.turbulence_model != 1 else ())
    print(f"[hand-off] {c.name} {c.nii}x{c.njj}", flush=True)
    got, ref = pf.run(c, iterations=4), pyoracle.run(c, iterations=4)
    for f, r in diff_report(got, ref, fields).items():
        assert r["n_bits_differ"] == 0, (c.name, f, r)


@pytest.mark.gpu
@pytest.mark.parametrize("model", [1, 2, 0])
def test_disjoint_rows(model):
    _check(_layout(model))


@pytest.mark.gpu
def test_city_with_such_columns():
    _check(domain.build_case("handcity", 200, 190, domain.city_buildings(200, 190, 2.0, 2), dx=2.0, vertcellsff=16, speed10=4.0,
                             direction=235.0, z0=0.5, iterations=4))
