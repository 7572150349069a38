"""Global means over a block's load rounds: part-filled and several of them,
fields that start on 16 bytes and on 8."""
import numpy as np
import pytest

import oracle
import shtamd

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,im,jm", [(0, 16, 2), (7, 16, 10), (21, 64, 32), (31, 64, 48), (85, 256, 128), (170, 512, 256)])
@pytest.mark.parametrize("shift", [0, 1])
def test_avr_against_oracle(N, im, jm, shift):
    nf = 3
    g = 200.0 + np.random.default_rng(im + jm).standard_normal((nf, jm, im))
    buf = torch.empty(nf * jm * im + 2, dtype=torch.float64, device="cuda")
    v = buf[shift:shift + nf * jm * im]
    v.copy_(torch.from_numpy(g).cuda().reshape(-1))
    avg = torch.empty(nf, dtype=torch.float64, device="cuda")
    p = shtamd.Plan(N, im, jm, nf)
    p.avr_lonlat(v, avg, nf)
    torch.cuda.synchronize()
    # im jm terms of size 200 summed in another order: 512 x 256 of them stay within 2e-12 of each other
    assert np.abs(avg.cpu().numpy() - oracle.Plan(N, im, jm).avr_lonlat(g)).max() < 2e-12
    p.close()


@pytest.mark.parametrize("N,im,jm", [(40, 256, 64), (40, 256, 66), (5, 256, 512), (5, 1024, 126), (60, 2048, 62)])
@pytest.mark.parametrize("shift", [0, 1])
def test_avr_of_several_rounds(N, im, jm, shift):
    """Fields of one full round and a little more, of a part-filled last round, of
    the most rows: against the oracle, at most 512 x 256 terms as above."""
    test_avr_against_oracle(N, im, jm, shift)


@pytest.mark.parametrize("N,im,jm", [(42, 128, 64), (85, 256, 128), (106, 512, 160), (170, 512, 256)])
def test_avr_rounding_errors(N, im, jm):
    """The sum is a tree over threads and waves.  One addition rounds by 0.46e-16 rms (a uniform
    half ulp over the mantissas); a tree's last levels add up to sqrt(1 + 1/2 + 1/4 + ...) of
    these, the division by 2 im one more: 0.8e-16.  Sixteen waves' sums added in a row have
    sqrt(2^2 + ... + 16^2) / 16 = 2.4 instead: 1.2e-16."""
    nf = 400
    mid = np.linspace(-0.5, 0.5, jm) * np.pi
    g = 2.0 * np.random.default_rng(1).standard_normal((nf, jm, im)) + (200.0 + 100.0 * np.cos(mid) ** 2)[None, :, None]
    p = shtamd.Plan(N, im, jm, nf)
    w = np.asarray(p.grid()[3])
    avg = torch.empty(nf, dtype=torch.float64, device="cuda")
    p.avr_lonlat(torch.from_numpy(g).cuda(), avg, nf)
    ref = (g.astype(np.longdouble).sum(-1) * w.astype(np.longdouble)).sum(-1) / (2 * im)
    err = ((avg.cpu().numpy() - ref) / ref).astype(float)
    assert np.sqrt((err * err).mean()) < 1.05e-16
    p.close()
