"""SPML packing, its inverse and the Laplacian powers over part-filled field
groups, degrees longer than a load round and the largest truncation; arrays
that start on 8 bytes."""
import numpy as np
import pytest

import oracle
import shtamd
from shtamd import synth

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def shifted(a, shift):
    """a on the device, starting `shift` doubles into an allocation."""
    buf = torch.empty(a.size + 2, dtype=torch.float64, device="cuda")
    v = buf[shift:shift + a.size]
    v.copy_(torch.from_numpy(np.ascontiguousarray(a)).cuda().reshape(-1))
    return v


@pytest.mark.parametrize("N,im,jm", [(0, 16, 2), (1, 16, 2), (21, 64, 32), (42, 128, 64), (85, 256, 128), (255, 512, 256)])
@pytest.mark.parametrize("nf,shift", [(1, 0), (8, 1), (19, 0)])
def test_pack_and_laplacian(N, im, jm, nf, shift):
    s = synth.spectra(N, nf, cfg=8)
    s[0] = np.arange(1, nf + 1)
    p = shtamd.Plan(N, im, jm, nf)
    spec, wa = shifted(shtamd.spec_to_real(s), shift), shifted(np.full((nf, (N + 1) ** 2), np.nan), shift)
    p.canon_to_spml(spec, wa, nf)
    want = oracle.spml_pack(s, N)
    # one product by sqrt(2) on either side
    assert np.abs(wa.cpu().numpy().reshape(nf, -1) - want).max() <= 4e-16 * np.abs(want).max()
    back = torch.full_like(spec, np.nan)
    p.spml_to_canon(wa, back, nf)
    got = shtamd.real_to_spec(back.cpu().numpy().reshape(-1, nf, 2))
    assert np.abs(got - s).max() <= 8e-16 * np.abs(s).max()
    for power in (-2, 1, 4):
        out = torch.full_like(back, np.nan)[: 2 * p.K * nf]
        a = back.clone()  # 16-byte aligned
        p.spec_lapla(a, out, power, nf)
        ref = oracle.spec_lapla(got, N, power)
        # up to four products or divisions on either side
        assert np.abs(shtamd.real_to_spec(out.cpu().numpy().reshape(-1, nf, 2)) - ref).max() <= 2e-15 * np.abs(ref).max()
        p.spec_lapla(a, a, power, nf)
        assert torch.equal(a, out)
    p.close()


@pytest.mark.parametrize("N,im,jm,nf", [(10, 32, 16, 3031), (21, 64, 32, 800), (42, 128, 64, 9), (42, 128, 64, 70), (85, 256, 128, 18), (255, 512, 256, 9)])
def test_pack_both_sides_of_the_line(N, im, jm, nf):
    """Calls large enough for the tiles: bitwise what small calls of the same fields give."""
    rng = np.random.default_rng(N)
    p = shtamd.Plan(N, im, jm, nf)
    wa = torch.from_numpy(rng.standard_normal((nf, (N + 1) ** 2))).cuda()
    spec, back = torch.full((p.K, nf, 2), np.nan, dtype=torch.float64, device="cuda"), torch.full_like(wa, np.nan)
    p.spml_to_canon(wa, spec, nf)
    p.canon_to_spml(spec, back, nf)
    for f in (0, 7, nf - 1):
        s1, w1 = torch.full((p.K, 1, 2), np.nan, dtype=torch.float64, device="cuda"), torch.full_like(wa[:1], np.nan)
        p.spml_to_canon(wa[f:f + 1].clone(), s1, 1)
        p.canon_to_spml(s1, w1, 1)
        assert torch.equal(spec[:, f:f + 1], s1) and torch.equal(back[f:f + 1], w1), f
    p.close()
