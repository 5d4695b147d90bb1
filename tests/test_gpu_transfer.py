"""Transfers between the device and the caller's arrays, in chunks through the
pinned ring: fields of less than one piece, of one chunk and of several (a chunk
holds 8 MB, a piece 256 KB), and a file of several chunks.  Every value
arrives, bit for bit, and levels the device does not hold pass through."""
import numpy as np
import pytest

from gral_amd import domain


@pytest.mark.gpu
@pytest.mark.parametrize("nii,njj,vcf", [(9, 8, 8), (64, 61, 30), (231, 229, 40)])
def test_fields_round_trip(nii, njj, vcf):
    from gral_amd import pf
    bl = [domain.Building(3, 4, 3, 5, 6.5)]
    c = domain.build_case("mv", nii, njj, bl, dx=2.0, vertcellsff=vcf, direction=235.0, iterations=4)
    rng = np.random.default_rng(5)
    x = {f: rng.standard_normal(c.uk.shape, dtype=np.float32) for f in ("uk", "vk", "wk")}
    print(f"[transfer] {nii}x{njj}, {c.kadvmax + 2} of {c.nkk + 2} levels on the device", flush=True)
    with pf.PrognosticFlowfield(c) as s:
        s.prepare(iterations=4)
        s.momentum_sweep(2)
        s.restore_ckpt()                                  # the device's fields are the newer ones from here
        s.set_velocity(x["uk"], x["vk"], x["wk"])
        a = s.download()
        s.forward_ckpt(1)
        s.restore_ckpt()
        b = s.download()
        s.momentum_sweep(2)
        g = s.momentum_vjp(x["wk"])
    up = c.kadvmax + 2
    assert np.array_equal(g[:, :, up:].view(np.uint32), x["wk"][:, :, up:].view(np.uint32))
    for f in x:
        assert np.array_equal(a[f].view(np.uint32), x[f].view(np.uint32)), f
        assert np.array_equal(b[f].view(np.uint32), x[f].view(np.uint32)), f


@pytest.mark.gpu
def test_file_of_several_chunks():
    # 26 MB: the records of two builds of the file are the same, and its values are the fields' times 100
    from gral_amd import pf
    c = domain.build_case("mf", 140, 139, [domain.Building(3, 4, 3, 5, 6.5)], dx=2.0, vertcellsff=12, direction=235.0, iterations=2)
    with pf.PrognosticFlowfield(c) as s:
        s.prepare(iterations=2)
        s.iterate(2)
        n = s.gff_size(0)
        buf = np.zeros(n, np.uint8)
        s.gff_payload_into(0, buf)
        f = s.download()
    assert n > 24 << 20
    v = buf[32:].view(np.int16).reshape(c.nii + 1, c.njj + 1, c.nkk + 1, 3)
    want = (f["uk"][1:c.nii + 2, 1:c.njj + 2, :c.nkk + 1] * np.float32(100.0)).astype(np.int16)
    assert np.array_equal(v[..., 0], want)
