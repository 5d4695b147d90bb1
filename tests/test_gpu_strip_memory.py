"""A tall situation that took the strips' buffers gives them back when a later call on it
needs the memory: within a budget of device memory that holds its fields and the
adjoint's, but not the strips' beside them, the window and its VJP run, per-diagonal from
there on, with the results of a handle without a budget."""
import numpy as np
import pytest

from tests.helpers import FIELDS, diff_report
from tests.test_gpu_strips import _city


@pytest.mark.gpu
@pytest.mark.parametrize("graph", ["0", "1"])
def test_strips_make_room_for_the_adjoint(monkeypatch, graph):
    from gral_amd import pf
    monkeypatch.setenv("GRAL_PF_GRAPH", graph)
    c = _city(16, 15, 50, tower=118.0)                    # 0.18 MB a field: 12 of the solver, 19 of the strips, 15 of the adjoint
    g = [np.random.default_rng(q).standard_normal(c.uk.shape).astype(np.float32) for q in range(3)]
    out = []
    for mb in (None, 6):
        if mb:
            monkeypatch.setenv("GRAL_PF_DEVICE_MB", str(mb))
        with pf.PrognosticFlowfield(c) as s:
            print(f"[strip memory] budget {mb} MB graph {graph}", flush=True)
            s.prepare(20)
            for _ in range(2):                            # the second one replays the captured chunk
                s.iterate(4)
                assert s.timing()["launches"] < 200
            s.forward_ckpt(3)
            v = s.vjp(*g)
            s.restore_ckpt()
            s.iterate(4)
            assert (s.timing()["launches"] > 200) == (mb is not None)
            out.append((v, s.download()))
    for a, b in zip(out[0][0], out[1][0]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    for f, r in diff_report(out[1][1], out[0][1], FIELDS).items():
        assert r["n_bits_differ"] == 0, (f, r)
