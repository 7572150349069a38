"""The transform workloads whose speed is tracked, through the Python binding.

listed() names them, draw() gives more of the same ranges, prepare() builds the
plan and the inputs of one on the GPU, run() makes one pass, work() counts the
bytes and operations a pass cannot do without, exact() restates the pass in
64-bit torch on the CPU.

Ranges: triangular truncations up to N = 170 on Gaussian grids of 32 to 512
longitudes (a power of two), 1 to 776 fields a call, the four precision forms;
the zonal transform up to degree 1024; remaps between grids of up to 512 x 256
points.  Spectra fall off as n^-3 in variance; grids are temperatures of 200 to
300 K with 2 K of noise.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dennou-ccm_amd", "py"))
import shtamd  # noqa: E402

PRECISION = {"fp64": shtamd.PREC_FP64, "bf16x3": shtamd.PREC_SPLIT_BF16, "fp16": shtamd.PREC_SCALED_FP16,
             "bf16x6": shtamd.PREC_SPLIT_BF16X6}
GRIDS = {21: (64, 32), 42: (128, 64), 85: (256, 128), 170: (512, 256)}
LARGEST = 776 * 512 * 256  # grid points of the largest call


def _on(nmax, **more):
    im, jm = GRIDS[nmax]
    return {"nmax": nmax, "im": im, "jm": jm, **more}


def listed():
    return [
        # surface pressure of the T21 configurations to the grid: one field, launch latency
        _on(21, name="t21_surface", kind="synthesis", nf=1, prec="fp64"),
        # one time step's state of the T21L16 configuration: three variables on 16 levels and surface pressure
        _on(21, name="t21l16_state", kind="roundtrip", nf=49, prec="fp64"),
        # the dynamics' values and both gradients of the T42L26 state
        _on(42, name="t42l26_gradients", kind="gradients", nf=79, prec="fp64"),
        # the T85L32 state in the split form (the headline workload)
        _on(85, name="t85l32_state", kind="roundtrip", nf=97, prec="bf16x6"),
        # flux divergence of two tracers on 32 levels and one surface flux
        _on(85, name="t85l32_divergence", kind="divergence", nf=65, prec="fp64"),
        # the T170L48 state in double precision
        _on(170, name="t170l48_state", kind="roundtrip", nf=145, prec="fp64"),
        # the T170 members of an ensemble transformed as one batch
        _on(170, name="t170_members", kind="roundtrip", nf=776, prec="bf16x6"),
        # an ensemble of mixed truncations and level counts, one graph launch, scaled 16-bit form
        {"name": "ensemble", "kind": "ensemble", "t21": 3, "t42": 5, "t85": 4, "levels": 16, "prec": "fp16"},
        # the energy-balance model: one field of degree 1024, analysis and synthesis
        {"name": "ebm_zonal", "kind": "zonal", "nmax": 1024, "jm": 1024, "nf": 1},
        # coupler exchange: 12 fields of the T42 atmosphere to a 256 x 128 surface grid and their global means
        _on(85, name="coupler", kind="coupler", im_send=128, jm_send=64, nf=12),
        # hyperdiffusion tendency of a T85L32 state held in SPML's packing
        _on(85, name="t85l32_diffusion", kind="diffusion", nf=97, power=4),
        # what the Fortran model calls: host arrays in SPML's packing, 26 levels at T42, there and back
        _on(42, name="t42l26_host", kind="host", nf=26, prec="fp64"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng):
    """A truncation and a grid that holds it: the model's own, or any other."""
    if rng.random() < 0.5:
        return _on(rng.choice(sorted(GRIDS)))
    im = rng.choice([32, 64, 128, 256, 512])
    nmax = rng.randint(im // 5, (im - 1) // 3)
    jm = 2 * rng.randint(-(-(3 * nmax + 1) // 4), im // 2 - im // 16)
    return {"nmax": nmax, "im": im, "jm": jm}


def draw(rng):
    kind = rng.choice(["synthesis", "analysis", "roundtrip", "roundtrip", "gradients", "divergence", "ensemble",
                       "zonal", "coupler", "diffusion", "host"])
    if kind == "ensemble":
        return {"kind": kind, "t21": rng.randint(1, 8), "t42": rng.randint(1, 8), "t85": rng.randint(1, 6),
                "levels": rng.randint(4, 40), "prec": rng.choice(["fp64", "fp16", "bf16x6"])}
    if kind == "zonal":
        jm = 2 * _log(rng, 16, 512)
        return {"kind": kind, "nmax": rng.randint(jm // 2, jm), "jm": jm, "nf": _log(rng, 1, 97)}
    c = {"kind": kind, **_grid(rng)}
    most = min(776, LARGEST // (c["im"] * c["jm"]))
    if kind in ("gradients", "divergence", "host"):
        most //= 4  # several grids a call, or grids that pass through the host
    if kind == "coupler":
        im = rng.choice([32, 64, 128, 256])
        return {**c, "im_send": im, "jm_send": im // 2, "nf": _log(rng, 1, 40)}
    if kind == "diffusion":
        return {**c, "nf": _log(rng, 1, most), "power": rng.choice([-2, -1, 1, 2, 3, 4])}
    prec = "fp64" if kind in ("gradients", "divergence") else rng.choice(sorted(PRECISION))
    return {**c, "nf": _log(rng, 1, most // 2 if prec == "fp64" else most), "prec": prec}


# ---------------------------------------------------------------- inputs
def _degrees(nmax):
    """(n, m) of the canonical rows k = off(m) + n - m."""
    m = np.repeat(np.arange(nmax + 1), np.arange(nmax + 1, 0, -1))
    return np.arange(m.size) - (m * (nmax + 1) - m * (m - 1) // 2) + m, m


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _spectra(nmax, nf, gen):
    """Canonical (K, nf, 2): variance n^-3, real for m = 0, no mean."""
    n, m = (torch.from_numpy(a).cuda() for a in _degrees(nmax))
    amp = torch.where(n > 0, (0.5 * n.clamp(min=1).double() ** -3).sqrt(), 0.0)
    s = torch.randn((n.numel(), nf, 2), generator=gen, dtype=torch.float64, device="cuda") * amp[:, None, None]
    s[m == 0, :, 1] = 0.0
    return s


def _temperature(nf, jm, im, gen):
    mid = torch.linspace(-0.5, 0.5, jm, dtype=torch.float64, device="cuda") * math.pi
    g = torch.randn((nf, jm, im), generator=gen, dtype=torch.float64, device="cuda")
    return g.mul_(2.0).add_((200.0 + 100.0 * torch.cos(mid) ** 2)[None, :, None])


def _packed(nmax, nf, gen):
    """SPML's (nf, (N+1)^2) of spectra as above."""
    n = torch.from_numpy(np.repeat(np.arange(nmax + 1), 2 * np.arange(nmax + 1) + 1)).cuda()
    w = torch.randn((nf, n.numel()), generator=gen, dtype=torch.float64, device="cuda")
    return w.mul_(n.clamp(min=1).double() ** -1.5).mul_(n > 0)


def _bilinear(c):
    """Triplets of a bilinear remap between the latitude-longitude grids."""
    ims, jms, imd, jmd = c["im_send"], c["jm_send"], c["im"], c["jm"]
    y, x = (np.arange(jmd) + 0.5) / jmd * jms - 0.5, np.arange(imd) / imd * ims
    j0, i0 = np.floor(y).astype(np.int64), np.floor(x).astype(np.int64)
    fy, fx = y - j0, x - i0
    si, cf = [], []
    for dj, wy in ((0, 1 - fy), (1, fy)):
        for di, wx in ((0, 1 - fx), (1, fx)):
            si.append(np.clip(j0 + dj, 0, jms - 1)[:, None] * ims + ((i0 + di) % ims)[None, :])
            cf.append(wy[:, None] * wx[None, :])
    ri = np.broadcast_to(np.arange(imd * jmd), (4, imd * jmd))
    return (np.stack(si).reshape(4, -1).T.ravel().astype(np.int32), ri.T.ravel().astype(np.int32),
            np.stack(cf).reshape(4, -1).T.ravel())


def _members(c):
    out = []
    for nmax in (21, 42, 85):
        for j in range(c["t%d" % nmax]):
            out.append((nmax, *GRIDS[nmax], 3 * max(1, c["levels"] * (j + 1) // (j + 2)) + 1))
    return out


def _inputs(c, gen):
    kind = c["kind"]
    if kind in ("synthesis", "roundtrip", "gradients"):
        return [_spectra(c["nmax"], c["nf"], gen)]
    if kind == "analysis":
        return [_temperature(c["nf"], c["jm"], c["im"], gen)]
    if kind == "divergence":
        return [_temperature(c["nf"], c["jm"], c["im"], gen).sub_(250.0) for _ in range(2)]
    if kind == "ensemble":
        return [_spectra(m[0], m[3], gen) for m in _members(c)]
    if kind == "zonal":
        lat = torch.linspace(-0.5, 0.5, c["jm"], dtype=torch.float64, device="cuda") * math.pi
        return [300.0 - 60.0 * torch.sin(lat) ** 2 + torch.randn((c["nf"], c["jm"]), generator=gen, dtype=torch.float64, device="cuda")]
    if kind == "coupler":
        return [_temperature(c["nf"], c["jm_send"], c["im_send"], gen)]
    return [_packed(c["nmax"], c["nf"], gen)]  # diffusion, host


class _Buffer:
    """A device buffer of a batch as torch.as_tensor takes it; it keeps the batch."""

    def __init__(self, batch, ptr, shape, strides):
        self.batch = batch
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "strides": strides, "typestr": "<f8", "version": 3}


def _view(batch, ptr, shape, strides):
    """Tensor over a batch's buffer.  The memory is the batch's and goes with it, so the tensor
    holds the batch: results may be read after the state that ran it is gone."""
    t = torch.as_tensor(_Buffer(batch, ptr, shape, strides), device="cuda")
    t.batch = batch
    return t


def _empty(*shape):
    return torch.empty(shape, dtype=torch.float64, device="cuda")


def prepare(case, seed):
    c = case
    inp = _inputs(c, _generator(seed))
    s = {"case": c, "in": inp}
    kind, nf = c["kind"], c.get("nf")
    if kind == "ensemble":
        s["batch"] = b = shtamd.Batch(_members(c), precision=PRECISION[c["prec"]])
        s["out"] = []
        for j, ((nmax, im, jm, k), x) in enumerate(zip(_members(c), inp)):
            spec_in, grid, spec_out, ld = b.member_ptrs(j)
            rows = shtamd.ncoef(nmax)
            views = [_view(b, p, (rows, k, 2), (8 * ld, 16, 8)) for p in (spec_in, spec_out)]
            views[0].copy_(x)
            s["out"] += [_view(b, grid, (k, jm, im), (8 * jm * im, 8 * im, 8)), views[1]]
        return s
    if kind == "zonal":
        s["zonal"] = shtamd.Zonal(c["nmax"], c["jm"], nf)
        s["out"] = [_empty(nf, c["nmax"] + 1), _empty(nf, c["jm"])]
        return s
    flags = shtamd.FLAG_GRAD if kind in ("gradients", "divergence") else 0
    s["plan"] = p = shtamd.Plan(c["nmax"], c["im"], c["jm"], nf, precision=PRECISION[c.get("prec", "fp64")], flags=flags)
    grid, spec = (nf, c["jm"], c["im"]), (p.K, nf, 2)
    if kind == "host":
        s["in"] = [inp[0].cpu().numpy()]
        s["out"] = [np.empty(grid), np.empty(s["in"][0].shape)]
    elif kind == "coupler":
        si, ri, cf = _bilinear(c)
        s["remap"] = shtamd.Remap(si, ri, cf, c["im_send"] * c["jm_send"], c["im"] * c["jm"])
        s["out"] = [_empty(*grid), _empty(nf)]
    elif kind == "diffusion":
        s["out"] = [_empty(*spec), _empty(*spec), _empty(*inp[0].shape)]
    else:
        s["out"] = {"synthesis": [grid], "analysis": [spec], "roundtrip": [grid, spec], "gradients": [grid] * 3, "divergence": [spec]}[kind]
        s["out"] = [_empty(*x) for x in s["out"]]
    return s


# ---------------------------------------------------------------- one pass
def run(state):
    c, x, out = state["case"], state["in"], state["out"]
    kind, nf = c["kind"], c.get("nf")
    if kind == "ensemble":
        state["batch"].run(shtamd.DIR_ROUNDTRIP)
        return out
    if kind == "zonal":
        state["zonal"].l_y_dev(x[0], out[0], nf)
        state["zonal"].y_l_dev(out[0], out[1], nf)
        return out
    p = state["plan"]
    if kind == "synthesis":
        p.spec_to_grid(x[0], out[0], nf)
    elif kind == "analysis":
        p.grid_to_spec(x[0], out[0], nf)
    elif kind == "roundtrip":
        p.spec_to_grid(x[0], out[0], nf)
        p.grid_to_spec(out[0], out[1], nf)
    elif kind == "gradients":
        p.spec_to_grad(x[0], *out, nf)
    elif kind == "divergence":
        p.grid_to_div(x[0], x[1], out[0], nf)
    elif kind == "coupler":
        state["remap"].apply(x[0], out[0], nf)
        p.avr_lonlat(out[0], out[1], nf)
    elif kind == "diffusion":
        p.spml_to_canon(x[0], out[0], nf)
        p.spec_lapla(out[0], out[1], c["power"], nf)
        p.canon_to_spml(out[1], out[2], nf)
    else:
        p.xya_wa(x[0], out[0])
        p.wa_xya(out[0], out[1])
    return out


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    c, kind = case, case["kind"]
    if kind == "ensemble":
        return _sum(_transform(*m, 2, 1) for m in _members(c))
    if kind == "zonal":
        n, jm, nf = c["nmax"] + 1, c["jm"], c["nf"]
        # either direction: the table of one hemisphere, every field in and out
        return {"bytes": 2 * (8 * n * (jm // 2) + 8 * nf * (n + jm)), "flops": 2 * (2 * n * (jm // 2) * nf)}
    nmax, im, jm, nf = c["nmax"], c["im"], c["jm"], c["nf"]
    grid = 8 * im * jm * nf
    if kind == "coupler":
        nnz, nsend = 4 * im * jm, c["im_send"] * c["jm_send"]
        return {"bytes": 12 * nnz + 8 * nsend * nf + 2 * grid + 8 * nf, "flops": 2 * nnz * nf + 2 * im * jm * nf}
    if kind == "diffusion":
        wa, spec = 8 * (nmax + 1) ** 2 * nf, 16 * shtamd.ncoef(nmax) * nf
        return {"bytes": 2 * wa + 4 * spec, "flops": 2 * shtamd.ncoef(nmax) * nf}
    if kind == "host":
        return _transform(nmax, im, jm, nf, 2, 1)
    one = {"synthesis": (1, 1), "analysis": (1, 1), "roundtrip": (2, 1), "gradients": (1, 3), "divergence": (1, 2)}[kind]
    return _transform(nmax, im, jm, nf, *one)


def _transform(nmax, im, jm, nf, passes, grids):
    """Passes between one set of spectra and `grids` grids: with two or more grids one carries the
    derivative table, the others share a Legendre sum."""
    K = shtamd.ncoef(nmax)
    tables = 1 if grids == 1 else 2
    fft = 2.5 * jm * im * math.log2(im) * nf
    return {"bytes": passes * (8 * im * jm * nf * grids + 16 * K * nf + 8 * K * (jm // 2) * tables),
            "flops": int(passes * (2 * jm * K * nf * tables + fft * grids))}


def _sum(parts):
    parts = list(parts)
    return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}


# ---------------------------------------------------------------- the same in 64 bits, without the library
def _gauss(jm):
    """Gauss nodes south to north and weights (sum 2), by Newton from the Chebyshev-like guess."""
    x = -np.cos(np.pi * (np.arange(jm) + 0.75) / (jm + 0.5))
    for _ in range(6):
        a, b = np.ones_like(x), x.copy()
        for n in range(2, jm + 1):
            a, b = b, ((2 * n - 1) * x * b - (n - 1) * a) / n
        d = jm * (a - x * b) / (1 - x * x)
        x = x - b / d
    return torch.from_numpy(x), torch.from_numpy(2 / ((1 - x * x) * d * d))


def _eps(n, m):
    return math.sqrt((n * n - m * m) / (4.0 * n * n - 1.0)) if n > 0 else 0.0


class _Exact:
    def __init__(self, nmax, im, jm):
        self.nmax, self.im, self.jm = nmax, im, jm
        self.mu, self.w = _gauss(jm)
        self.cos = torch.sqrt((1 - self.mu) * (1 + self.mu))
        sectoral = torch.ones(jm, dtype=torch.float64)
        self.P, self.H = [], []  # per m (jm, N - m + 1): Pt and (1 - mu^2) dPt/dmu
        for m in range(nmax + 1):
            if m:
                sectoral = sectoral * self.cos * math.sqrt((2 * m + 1) / (2.0 * m))
            col = [torch.zeros_like(sectoral), sectoral]
            for n in range(m, nmax + 1):
                col.append((self.mu * col[-1] - _eps(n, m) * col[-2]) / _eps(n + 1, m))
            self.P.append(torch.stack(col[1:-1], 1))
            self.H.append(torch.stack([(n + 1) * _eps(n, m) * col[n - m] - n * _eps(n + 1, m) * col[n - m + 2]
                                       for n in range(m, nmax + 1)], 1))

    def rows(self, m):
        o = m * (self.nmax + 1) - m * (m - 1) // 2
        return slice(o, o + self.nmax + 1 - m)

    def synthesis(self, spec, kind=0):
        """kind 0 value, 1 GradLon, 2 GradLat of (K, nf, 2) spectra."""
        nf = spec.shape[1]
        four = torch.zeros((nf, self.jm, self.im // 2 + 1), dtype=torch.complex128)
        for m in range(self.nmax + 1):
            s = spec[self.rows(m)].reshape(-1, 2 * nf)
            f = torch.view_as_complex(((self.H if kind == 2 else self.P)[m] @ s).reshape(self.jm, nf, 2))
            four[:, :, m] = (f * 1j * m if kind == 1 else f).T
        g = torch.fft.irfft(four, n=self.im) * self.im
        return g / self.cos[None, :, None] if kind else g

    def _quadrature(self, four, tables):
        """four (nf, jm, im/2+1) with the weights folded in."""
        out = torch.empty((shtamd.ncoef(self.nmax), four.shape[0], 2), dtype=torch.float64)
        for m in range(self.nmax + 1):
            f = torch.view_as_real(four[:, :, m].T.contiguous()).reshape(self.jm, -1)
            out[self.rows(m)] = (tables[m].T @ f).reshape(-1, four.shape[0], 2)
        return out

    def _fourier(self, grid, scale):
        return torch.fft.rfft(grid) * (0.5 / self.im * self.w * scale)[None, :, None]

    def analysis(self, grid):
        return self._quadrature(self._fourier(grid, 1.0), self.P)

    def divergence(self, a, b):
        im_m = 1j * torch.arange(self.im // 2 + 1, dtype=torch.float64)
        fa, fb = self._fourier(a, 1 / self.cos) * im_m, self._fourier(b, -1 / self.cos)
        return self._quadrature(fa, self.P) + self._quadrature(fb, self.H)


def _root2(m):
    return torch.where(m > 0, 2.0, 1.0).double().sqrt()


def _unpack(wa, nmax):
    """SPML's packing (nf, (N+1)^2) to canonical (K, nf, 2)."""
    n, m = (torch.from_numpy(a) for a in _degrees(nmax))
    re, im = wa[:, n * (n + 1) + m] / _root2(m), torch.where(m > 0, -wa[:, n * (n + 1) - m] / math.sqrt(2.0), 0.0)
    return torch.stack([re.T, im.T], -1)


def _pack(spec, nmax):
    n, m = (torch.from_numpy(a) for a in _degrees(nmax))
    wa = torch.empty((spec.shape[1], (nmax + 1) ** 2), dtype=torch.float64)
    wa[:, n * (n + 1) - m] = (-math.sqrt(2.0) * spec[:, :, 1]).T
    wa[:, n * (n + 1) + m] = (_root2(m)[:, None] * spec[:, :, 0]).T
    return wa


def _zonal_exact(c, y):
    mu, w = _gauss(c["jm"])
    col = [torch.zeros_like(mu), torch.ones_like(mu)]
    for n in range(c["nmax"] + 1):
        col.append((mu * col[-1] - _eps(n, 0) * col[-2]) / _eps(n + 1, 0))
    P = torch.stack(col[1:-1], 1)
    if c["nmax"] == c["jm"]:
        P[:, -1] = 0.0  # degree jm vanishes at every node
    lc = (y * (0.5 * w)) @ P
    return [lc, lc @ P.T]


def exact(case, seed):
    c, kind = case, case["kind"]
    x = [t.cpu() for t in _inputs(c, _generator(seed))]
    if kind == "zonal":
        return _zonal_exact(c, x[0])
    if kind == "diffusion":
        n = torch.from_numpy(_degrees(c["nmax"])[0]).double()
        fac = torch.where(n > 0, (-(n * (n + 1)).clamp(min=1)) ** c["power"], 0.0)
        spec = _unpack(x[0], c["nmax"])
        out = spec * fac[:, None, None]
        return [spec, out, _pack(out, c["nmax"])]
    if kind == "coupler":
        si, ri, cf = (torch.from_numpy(a) for a in _bilinear(c))
        flat = x[0].reshape(c["nf"], -1)
        g = (flat[:, si.long()] * cf).reshape(c["nf"], -1, 4).sum(-1).reshape(c["nf"], c["jm"], c["im"])
        return [g, (g.mean(-1) * (0.5 * _gauss(c["jm"])[1])).sum(-1)]
    if kind == "ensemble":
        ref, out = {}, []
        for (nmax, im, jm, _), s in zip(_members(c), x):
            e = ref.setdefault(nmax, None) or _Exact(nmax, im, jm)
            ref[nmax] = e
            g = e.synthesis(s)
            out += [g, e.analysis(g)]
        return out
    e = _Exact(c["nmax"], c["im"], c["jm"])
    if kind == "host":
        g = e.synthesis(_unpack(x[0], c["nmax"]))
        return [g, _pack(e.analysis(g), c["nmax"])]
    if kind == "analysis":
        return [e.analysis(x[0])]
    if kind == "divergence":
        return [e.divergence(*x)]
    if kind == "gradients":
        return [e.synthesis(x[0], k) for k in range(3)]
    g = e.synthesis(x[0])
    return [g] if kind == "synthesis" else [g, e.analysis(g)]
