"""Downloads in parts, between other calls: a field that the device changed reaches the
caller and the handle's own copy at once, whichever fields are asked for and in which
order, and what is not asked for stays newer on the device until a call needs it."""
import ctypes as C

import numpy as np
import pytest

from gral_amd import domain
from tests.helpers import FIELDS, KE_FIELDS

NAMES = ("uk", "vk", "wk", "uks", "vks", "wks", "dpm", "dpmnew", "turb", "tdiss")


def _part(s, names):
    out = {f: np.full(s.case.uk.shape, np.nan, np.float32) for f in names}
    a = [out[f].ctypes.data_as(C.POINTER(C.c_float)) if f in out else None for f in NAMES]
    assert s.lib.gral_pf_download_fields(s.h, *a) == 0
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("model", [1, 2])
def test_parts(model):
    from gral_amd import pf
    bl = domain.city_buildings(40, 37, 2.0, 3, density=0.2, fmin=4.0, fmax=12.0, hmin=3.0, hmax=14.0, margin=2)
    c = domain.build_case("dl", 40, 37, bl, dx=2.0, vertcellsff=12, speed10=4.0, direction=215.0, z0=0.5, turbulence_model=model,
                          iterations=20)
    fields = list(FIELDS + (KE_FIELDS if model != 1 else ()))
    parts = [["uk"], ["vks", "wk"], fields[::-1], ["dpm", "vks"], fields, fields]
    with pf.PrognosticFlowfield(c) as s, pf.PrognosticFlowfield(c) as r:
        s.prepare(20)
        r.prepare(20)
        for names in parts:
            for other in (None, "finish", "set_velocity", "diagnostic"):
                print(f"[download] model {model}, {len(names)} fields, then {other}", flush=True)
                s.iterate(1)
                r.iterate(1)
                r.finish()                                # all host copies from the device
                ref = r.download()
                for f, a in _part(s, names).items():
                    assert np.array_equal(a.view(np.uint32), ref[f].view(np.uint32)), (names, f)
                if other == "finish":
                    assert s.finish()["unreal_u"] == r.finish()["unreal_u"]
                elif other == "set_velocity":
                    v = [0.9 * ref[f] for f in ("uk", "vk", "wk")]
                    s.set_velocity(*v)
                    r.set_velocity(*v)
                elif other == "diagnostic":
                    s.diagnostic(1)
                    r.diagnostic(1)
                ref = r.download()
                for got in (_part(s, fields[::2]), _part(s, fields), _part(s, fields)):
                    for f, a in got.items():
                        assert np.array_equal(a.view(np.uint32), ref[f].view(np.uint32)), (names, other, f)
