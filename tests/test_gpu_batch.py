"""Ensemble batches (sht_batch_*): members of uneven truncation and level count
in shared launches and graph branches.  Each member's result must be bitwise the same as the same
member transformed alone, and match the FP64 oracle (1e-12, or the mixed
form's tolerance); graph replays must equal the eager run every time."""
import numpy as np
import pytest

import oracle
import shtamd
from shtamd import hipmem, synth

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

GRIDS = {21: (64, 32), 42: (128, 64), 85: (256, 128)}
MEMBERS = [(21, 16), (42, 13), (85, 10), (42, 7), (21, 5), (85, 3), (42, 1)]  # (N, nfield)


def rel(a, b):
    return float(np.linalg.norm(np.ravel(a - b)) / np.linalg.norm(np.ravel(b)))


def make_batch(prec):
    descs = [(N, *GRIDS[N], nf) for (N, nf) in MEMBERS]
    b = shtamd.Batch(descs, precision=prec)
    specs = []
    for j, (N, nf) in enumerate(MEMBERS):
        s = synth.spectra(N, nf, cfg=3, member=j)
        spec_in, grid, spec_out, ld = b.member_ptrs(j)
        hipmem.put_member_spectra(spec_in, ld, s)
        specs.append(s)
    return b, specs


def read_member(b, j):
    N, nf = MEMBERS[j]
    im, jm = GRIDS[N]
    spec_in, grid, spec_out, ld = b.member_ptrs(j)
    K = (N + 1) * (N + 2) // 2
    return hipmem.from_device(grid, (nf, jm, im)), hipmem.get_member_spectra(spec_out, ld, K, nf)


@pytest.mark.parametrize("prec,tol", [(shtamd.PREC_FP64, 1e-12), (shtamd.PREC_SPLIT_BF16X6, 1e-6)])
def test_batch_matches_alone_and_oracle(prec, tol):
    b, specs = make_batch(prec)
    b.run_eager(shtamd.DIR_ROUNDTRIP)
    torch.cuda.synchronize()
    for j, (N, nf) in enumerate(MEMBERS):
        im, jm = GRIDS[N]
        g, s_rt = read_member(b, j)
        ref = oracle.Plan(N, im, jm)
        assert rel(g, ref.spec_to_grid(specs[j])) < tol, j
        assert rel(s_rt, specs[j]) < 2 * tol, j
        # the same member alone through a plan of its own: bitwise equal
        p = shtamd.Plan(N, im, jm, nf, precision=prec)
        si = torch.from_numpy(shtamd.spec_to_real(specs[j])).cuda()
        ga = torch.empty((nf, jm, im), dtype=torch.float64, device="cuda")
        so = torch.empty_like(si)
        p.spec_to_grid(si, ga, nf)
        p.grid_to_spec(ga, so, nf)
        torch.cuda.synchronize()
        assert np.array_equal(ga.cpu().numpy(), g), j
        assert np.array_equal(shtamd.real_to_spec(so.cpu().numpy()), s_rt), j
        p.close()
    b.close()


def test_batch_graph_replays_equal_eager():
    b, specs = make_batch(shtamd.PREC_FP64)
    b.run_eager(shtamd.DIR_ROUNDTRIP)
    torch.cuda.synchronize()
    ref = [read_member(b, j) for j in range(len(MEMBERS))]
    scratch = torch.zeros(1 << 20, dtype=torch.float64, device="cuda")
    for rep in range(4):
        # the program's own eager work between replays, and a fresh output state
        scratch.add_(1.0)
        for j in range(len(MEMBERS)):
            _, grid, spec_out, ld = b.member_ptrs(j)
            N, nf = MEMBERS[j]
            K = (N + 1) * (N + 2) // 2
            hipmem.put_member_spectra(spec_out, ld, np.zeros((K, nf), dtype=complex))
        b.run(shtamd.DIR_ROUNDTRIP)
        torch.cuda.synchronize()
        for j in range(len(MEMBERS)):
            g, s = read_member(b, j)
            assert np.array_equal(g, ref[j][0]) and np.array_equal(s, ref[j][1]), (rep, j)
    b.close()


def test_batch_inverse_forward_directions():
    b, specs = make_batch(shtamd.PREC_FP64)
    b.run(shtamd.DIR_INVERSE)
    torch.cuda.synchronize()
    for j, (N, nf) in enumerate(MEMBERS):
        im, jm = GRIDS[N]
        g, _ = read_member(b, j)
        assert rel(g, oracle.Plan(N, im, jm).spec_to_grid(specs[j])) < 1e-12
    b.run(shtamd.DIR_FORWARD)
    torch.cuda.synchronize()
    for j in range(len(MEMBERS)):
        _, s = read_member(b, j)
        assert rel(s, specs[j]) < 1e-12
    b.close()


def test_batch_autotune_keeps_results():
    """Autotuning a batch re-captures its graph with the tuned shapes; results
    stay within the FP64 bar and the graph still equals the eager run."""
    b, specs = make_batch(shtamd.PREC_FP64)
    b.autotune(reps=3)
    b.run(shtamd.DIR_ROUNDTRIP)
    torch.cuda.synchronize()
    graph_out = [read_member(b, j) for j in range(len(MEMBERS))]
    b.run_eager(shtamd.DIR_ROUNDTRIP)
    torch.cuda.synchronize()
    for j, (N, nf) in enumerate(MEMBERS):
        im, jm = GRIDS[N]
        g, s = read_member(b, j)
        assert np.array_equal(g, graph_out[j][0]) and np.array_equal(s, graph_out[j][1]), j
        assert rel(g, oracle.Plan(N, im, jm).spec_to_grid(specs[j])) < 1e-12, j
        assert rel(s, specs[j]) < 1e-12, j
    b.close()


MANY = [(7, 16, 10, 3), (5, 16, 8, 40), (10, 32, 16, 1), (9, 32, 26, 70), (21, 64, 32, 33), (20, 64, 48, 5),
        (31, 64, 64, 17), (42, 128, 64, 9), (50, 128, 100, 2), (85, 256, 128, 11), (100, 256, 202, 4), (0, 16, 2, 8)]


@pytest.mark.parametrize("prec", [shtamd.PREC_FP64, shtamd.PREC_SPLIT_BF16, shtamd.PREC_SCALED_FP16, shtamd.PREC_SPLIT_BF16X6])
@pytest.mark.parametrize("count", [2, len(MANY)])
def test_batch_shared_launches_bitwise(prec, count):
    """Two grids in one launch per stage, and more than a launch takes beside one
    of more latitude pairs: each direction bitwise as the member alone."""
    members = MANY[-count:] if count > 2 else MANY[4:6]
    b = shtamd.Batch(members, precision=prec)
    specs = [synth.spectra(N, nf, cfg=5, member=j) for j, (N, _, _, nf) in enumerate(members)]
    for j, s in enumerate(specs):
        spec_in, _, _, ld = b.member_ptrs(j)
        hipmem.put_member_spectra(spec_in, ld, s)
    for run in (b.run, b.run_eager):
        run(shtamd.DIR_INVERSE)
        run(shtamd.DIR_FORWARD)
        torch.cuda.synchronize()
        for j, (N, im, jm, nf) in enumerate(members):
            _, grid, spec_out, ld = b.member_ptrs(j)
            p = shtamd.Plan(N, im, jm, nf, precision=prec)
            si = torch.from_numpy(shtamd.spec_to_real(specs[j])).cuda()
            ga, so = torch.empty((nf, jm, im), dtype=torch.float64, device="cuda"), torch.empty_like(si)
            p.spec_to_grid(si, ga, nf)
            p.grid_to_spec(ga, so, nf)
            torch.cuda.synchronize()
            assert np.array_equal(hipmem.from_device(grid, (nf, jm, im)), ga.cpu().numpy()), j
            assert np.array_equal(hipmem.get_member_spectra(spec_out, ld, p.K, nf), shtamd.real_to_spec(so.cpu().numpy())), j
            p.close()
    b.close()


def test_batch_groups_beyond_one_launch():
    """Groups that fill a launch each (2^32 threads) do not share one: degree 0,
    every grid value is the field's coefficient, and it comes back."""
    nf = 9 << 20
    members = [(0, 16, 2, nf), (0, 16, 4, nf)]
    b = shtamd.Batch(members)
    rng = np.random.default_rng(3)
    vals = [rng.standard_normal(nf) for _ in members]
    for j, v in enumerate(vals):
        spec_in, _, _, ld = b.member_ptrs(j)
        hipmem.put_member_spectra(spec_in, ld, v[None, :].astype(complex))
    b.run(shtamd.DIR_ROUNDTRIP)
    torch.cuda.synchronize()
    for j, (_, im, jm, _) in enumerate(members):
        _, grid, spec_out, ld = b.member_ptrs(j)
        back = hipmem.get_member_spectra(spec_out, ld, 1, nf)[0]
        assert np.abs(back - vals[j]).max() < 1e-14, j
        for f0 in (0, nf // 2 - 500, nf - 1000):
            g = hipmem.from_device(grid + 8 * f0 * jm * im, (1000, jm * im))
            assert np.abs(g - vals[j][f0:f0 + 1000, None]).max() < 1e-14, (j, f0)
    b.close()


BIG = (100, 256, 202)  # more latitude pairs than a shared launch takes: a branch of its own


def round_trip_us(b, n=20):
    b.run(shtamd.DIR_ROUNDTRIP)
    best = float("inf")
    for _ in range(5):
        t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        t0.record()
        for _ in range(n):
            b.run(shtamd.DIR_ROUNDTRIP)
        t1.record()
        torch.cuda.synchronize()
        best = min(best, t0.elapsed_time(t1) / n * 1e3)
    return best


@pytest.mark.parametrize("prec", [shtamd.PREC_FP64, shtamd.PREC_SPLIT_BF16X6])
def test_batch_captured_graph_replays_and_is_dropped(prec):
    """A batch of shared and single groups runs as a graph: replays equal the eager run,
    and tuning after a capture keeps the members' data and gives a new graph that
    equals the eager run again."""
    members = [(21, 64, 32, 9), (42, 128, 64, 5), (*BIG, 6)]
    b = shtamd.Batch(members, precision=prec)
    specs = [synth.spectra(m[0], m[3], cfg=6, member=j) for j, m in enumerate(members)]

    def read():
        torch.cuda.synchronize()
        out = []
        for j, (N, im, jm, nf) in enumerate(members):
            _, grid, spec_out, ld = b.member_ptrs(j)
            out += [hipmem.from_device(grid, (nf, jm, im)), hipmem.get_member_spectra(spec_out, ld, shtamd.ncoef(N), nf)]
        return out

    def fill(which, value):
        for j, (N, im, jm, nf) in enumerate(members):
            spec_in, _, spec_out, ld = b.member_ptrs(j)
            hipmem.put_member_spectra(spec_in if which == "in" else spec_out, ld, specs[j] if value is None else np.full((shtamd.ncoef(N), nf), value, dtype=complex))

    scratch = torch.zeros(1 << 20, dtype=torch.float64, device="cuda")
    fill("in", None)
    for tuned in (False, True):
        b.run_eager(shtamd.DIR_ROUNDTRIP)
        ref = read()
        for rep in range(3):
            scratch.add_(1.0)
            fill("out", 7.0)
            b.run(shtamd.DIR_ROUNDTRIP)
            assert all(np.array_equal(x, y) for x, y in zip(read(), ref)), (tuned, rep)
        if not tuned:
            b.autotune(reps=2)
            assert all(np.array_equal(x, y) for x, y in zip(read(), ref))  # buffers untouched
    for j, (N, im, jm, nf) in enumerate(members):
        assert np.linalg.norm(ref[2 * j + 1] - specs[j]) / np.linalg.norm(specs[j]) < (1e-12 if prec == shtamd.PREC_FP64 else 2e-6)
    b.close()


@pytest.mark.parametrize("prec", [shtamd.PREC_FP64, shtamd.PREC_SCALED_FP16])
def test_batch_autotune_keeps_shared_launches(prec, tmp_path):
    """Groups whose tuned shape (here forced by a cache: K-split) is not the shared
    launches' stay in these where they are faster, as for small grids by far (20 us
    against 65 as graph branches): a tuned batch is not slower."""
    members = [(21, 64, 32, 49), (42, 128, 64, 40)]
    cache = tmp_path / "shapes.json"
    cache.write_text("{" + ", ".join(f'"T{N}_{im}x{jm}_nf{nf}_p{prec}": [0, 0, -1, -1, -1, -1]' for N, im, jm, nf in members) + "}")
    b = shtamd.Batch(members, precision=prec)
    before = round_trip_us(b)
    b.autotune(reps=3, cache_path=str(cache))
    after = round_trip_us(b)
    print(f"round trip {before:.1f} us, tuned {after:.1f} us", flush=True)
    assert after < 1.4 * before
    b.close()
