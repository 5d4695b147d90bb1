"""The particles' arrays on both sides of the sizes where their transfers change: one particle,
pageable copies, the pinned ring for the way up, and both ways (32 bytes of a particle go
to the device and 16 come back).  The wind at all of them is that of pieces of 50000."""
import numpy as np
import pytest

from gral_amd import domain


@pytest.mark.gpu
def test_counts():
    from gral_amd import pf
    c = domain.build_case("pt", 40, 37, [domain.Building(10, 15, 10, 14, 8.0)], dx=2.0, vertcellsff=12, direction=215.0, iterations=2)
    g = np.random.default_rng(2)
    n = 540000
    ci, cj = g.integers(2, 39, n).astype(np.int32), g.integers(2, 36, n).astype(np.int32)
    x, y = (ci - g.uniform(0, 1, n)) * 2.0, (cj - g.uniform(0, 1, n)) * 2.0
    z, ah = g.uniform(0.5, 15.0, n).astype(np.float32), np.zeros(n, np.float32)

    def wind(s, a, b):
        return s.wind_at_particles(1, 0, 0, 0.0, ci[a:b], cj[a:b], ah[a:b], x[a:b], y[a:b], z[a:b])

    with pf.PrognosticFlowfield(c) as s:
        s.prepare(2)
        s.iterate(2)
        parts = [wind(s, a, min(n, a + 50000)) for a in range(0, n, 50000)]
        ref = [np.concatenate(q) for q in zip(*parts)]
        for m in (1, 524000, 524288, 524289, n):
            print(f"[particles] {m}", flush=True)
            for got, r in zip(wind(s, 0, m), ref):
                assert np.array_equal(got.view(np.uint32), r[:m].view(np.uint32)), m
