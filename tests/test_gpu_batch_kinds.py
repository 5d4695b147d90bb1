"""Batches of tall situations with unlike sweeps: on strips, per-diagonal because the strips'
buffers found no memory, and per-diagonal because the columns have more levels than the
strips hold.  They are of one kind, run in one batch and give the plain solves' fields bit
for bit; a situation of at most 126 levels is refused beside them, as ever."""
import pytest

from tests.helpers import FIELDS, KE_FIELDS, diff_report
from tests.test_gpu_strips import _city


def _solver(pf, c, monkeypatch, mb=None):
    if mb:
        monkeypatch.setenv("GRAL_PF_DEVICE_MB", str(mb))
    s = pf.PrognosticFlowfield(c)
    monkeypatch.delenv("GRAL_PF_DEVICE_MB", raising=False)
    s.prepare(4)
    return s


def _diagonal(s):
    s.iterate(1)
    return s.timing()["launches"] > 50


@pytest.mark.gpu
@pytest.mark.parametrize("model,groups,graph", [(1, "1", "0"), (2, "2", "0"), (1, "1", "1")])
def test_mixed_batch(monkeypatch, model, groups, graph):
    from gral_amd import pf
    monkeypatch.setenv("GRAL_PF_GROUPS", groups)
    spec = [(dict(nii=16, njj=15, vcf=50, tower=118.0), None), (dict(nii=15, njj=16, vcf=49, tower=118.0), 4),
            (dict(nii=14, njj=13, vcf=62, tower=263.0, stretch=1.003), None), (dict(nii=14, njj=15, vcf=61, tower=263.0), None)]
    cases = [_city(model=model, direction=40.0 * q, **d) for q, (d, _) in enumerate(spec)]
    ref = []
    for c, (_, mb) in zip(cases, spec):
        print(f"[kinds] plain {c.name} {c.kadvmax + 2} levels", flush=True)
        with _solver(pf, c, monkeypatch, mb) as s:
            s.iterate(4)
            ref.append(s.download())
    monkeypatch.setenv("GRAL_PF_GRAPH", graph)
    sv = [_solver(pf, c, monkeypatch, mb) for c, (_, mb) in zip(cases, spec)]
    kinds = []
    for c, (_, mb) in zip(cases, spec):
        with _solver(pf, c, monkeypatch, mb) as s:
            kinds.append(_diagonal(s))
    assert kinds == [False, True, True, False]
    print(f"[kinds] batch model {model} groups {groups} graph {graph}", flush=True)
    with pf.Batch(sv) as b:
        for _ in range(2):
            b.iterate(2)
    for s, r in zip(sv, ref):
        for f, x in diff_report(s.download(), r, FIELDS + (KE_FIELDS if model != 1 else ())).items():
            assert x["n_bits_differ"] == 0, (s.case.name, f, x)
        s.close()


@pytest.mark.gpu
def test_mixed_stream(monkeypatch):
    from gral_amd import pf
    cases = [_city(16, 15, 50, tower=118.0), _city(14, 13, 62, tower=263.0, stretch=1.003)]
    sv = [_solver(pf, c, monkeypatch) for c in cases]
    with pf.Batch() as b:
        for s in sv:
            b.add(s)
        with _solver(pf, _city(16, 15, 50), monkeypatch) as low, pytest.raises(RuntimeError):
            b.add(low)
        assert len(b.step()) == 2                         # both at their iteration limit
    for s in sv:
        s.close()
