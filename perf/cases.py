"""The calls whose time is followed: what a user of the catalogue -> a_nlm transform has it do.

A case names a geometry (kmax, rmin, rmax, nside), a catalogue size and the entry point:

  cat      cat2amln of one catalogue (device arrays, or host arrays with "host")
  mocks    cat2amln_batch_device: several catalogues of one survey, uneven sizes
  vjp      the gradient of a scalar of a_nlm by radii and weights (field-level inference)
  field    field2anlm of a voxelised density field
  synth    anlm2field back to the voxels

The geometries are the configurations that the tests and bench.py run: 500-1000 Mpc/h at
nside 16-64 and 500-1500 Mpc/h at nside 64-256, kmax following the resolution, up to 4e6
galaxies.  Plans, windows and output buffers are made once, as a program that loops over
catalogues holds them.

Result types: an "fp64" plan's numbers are returned as they come.  A "mixed" plan's
coefficients and gradients are single-precision results in double-precision storage (its
precision is FP32 by choice of the caller), and the programs that choose it hold them as
what they are, in single precision.
"""
from __future__ import annotations

import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sphericalfourierbesseldecompositions.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import sfb_amd as S  # noqa: E402
from sfb_amd import _lib as L  # noqa: E402


def _case(name, kind, precision, kmax, rmin, rmax, nside, N, **more):
    c = {"name": name, "kind": kind, "precision": precision, "kmax": kmax, "rmin": rmin, "rmax": rmax,
         "nside": nside, "N": N, "weights": False, "window": "full", "host": False, "mocks": 1, "nr": 0}
    c.update(more)
    return c


def listed():
    return [
        # a first look at a small sample: numpy arrays in, numpy array out, the defaults
        _case("look_fp64_host", "cat", "fp64", 0.03, 500.0, 1000.0, 16, 20000, host=True),
        # the plain FP64 configuration: 1e5 galaxies, nside 32
        _case("shell32_fp64", "cat", "fp64", 0.05, 500.0, 1000.0, 32, 100000),
        # a weighted sample of odd size in a loop of fast transforms (likelihoods, mocks at low k)
        _case("shell32_mixed_weighted", "cat", "mixed", 0.05, 500.0, 1000.0, 32, 60013, weights=True, window="mask"),
        # a survey whose radial selection varies over the sky: dense window, weights, odd size
        _case("dense64_fp64", "cat", "fp64", 0.06, 500.0, 1000.0, 64, 300007, weights=True, window="dense"),
        # the headline size in the reference's precision, arrays resident on the GPU
        _case("shell128_fp64", "cat", "fp64", 0.1, 500.0, 1500.0, 128, 1000000),
        # the headline benchmark: one mixed-precision call from host arrays to host a_nlm
        _case("shell128_mixed_host", "cat", "mixed", 0.1, 500.0, 1500.0, 128, 1000000, host=True),
        # the large survey: northern hemisphere, Gaussian radial selection, weights
        _case("survey256_mixed", "cat", "mixed", 0.15, 500.0, 1500.0, 256, 4000000, weights=True, window="north"),
        # mock catalogues of uneven size through one plan
        _case("mocks128_mixed", "mocks", "mixed", 0.1, 500.0, 1500.0, 128, 500000, mocks=8),
        # gradients for field-level inference: FP64 on a medium sample, mixed at the headline size
        _case("grad64_fp64", "vjp", "fp64", 0.06, 500.0, 1000.0, 64, 200003, weights=True),
        _case("grad128_mixed", "vjp", "mixed", 0.1, 500.0, 1500.0, 128, 1000000),
        # a simulated density field to a_nlm, and a_nlm back to a field
        _case("field64_fp64", "field", "fp64", 0.06, 500.0, 1000.0, 64, 0, nr=75),
        _case("synth64_fp64", "synth", "fp64", 0.06, 500.0, 1000.0, 64, 0, nr=75),
    ]


def draw(rng):
    kind = rng.choice(["cat", "cat", "cat", "cat", "mocks", "vjp", "vjp", "field", "synth"])
    precision = "fp64" if kind in ("field", "synth") else rng.choice(["fp64", "mixed"])
    nside = rng.choice([16, 32, 64, 64, 128, 128] + ([256] if kind == "cat" and precision == "mixed" else []))
    rmin = round(rng.uniform(400.0, 700.0), 1)
    rmax = round(rng.uniform(900.0, 1600.0), 1)
    # lmax ~ kmax rmax runs from 0.6 to 1.15 nside (0.7 - 0.85 at nside 256, as the survey there)
    f = rng.uniform(0.6, 1.15) if nside < 256 else rng.uniform(0.7, 0.85)
    kmax = round(f * nside / rmax, 4)
    top = {16: 1e5, 32: 4e5, 64: 1e6, 128: 1e6, 256: 3e6}[nside]
    N = int(math.exp(rng.uniform(math.log(1e4), math.log(top)))) | rng.choice([0, 1])
    more = {}
    if kind == "cat":
        more["window"] = rng.choice(["full", "mask", "north"] + (["dense"] if nside <= 64 else []))
        more["host"] = rng.random() < 0.3
    if kind == "mocks":
        N = min(N, 400000)
        more["mocks"] = rng.randint(2, 6)
        more["window"] = rng.choice(["full", "mask"])
    if kind in ("field", "synth"):
        N, nside = 0, min(nside, 64)
        kmax = round(f * nside / rmax, 4)
        more["nr"] = rng.randint(20, 120)
    else:
        more["weights"] = rng.random() < 0.5
    c = _case("", kind, precision, kmax, rmin, rmax, nside, N, **more)
    del c["name"]
    return c


# ---- inputs: from the case and the seed alone -------------------------------------------


def _gen(seed, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _modes(case):
    return S.AnlmModes(case["kmax"], case["rmin"], case["rmax"], nside=case["nside"])


def _sizes(case, seed):
    """Galaxies of each catalogue: N, or uneven sizes around it for mocks."""
    if case["kind"] != "mocks":
        return [case["N"]]
    u = torch.rand(case["mocks"], dtype=torch.float64, generator=_gen(seed + 17, "cpu")).tolist()
    return [int(case["N"] * (0.2 + 1.6 * x)) for x in u]


def _selection(case, r):
    """Radial selection: Gaussian in the masked survey, else constant."""
    if case["window"] == "north":
        r0, sig = 0.5 * (case["rmin"] + case["rmax"]), 0.3 * (case["rmax"] - case["rmin"])
        return torch.exp(-((r - r0) ** 2) / (2 * sig * sig))
    return torch.ones_like(r)


def _catalogue(case, n, seed):
    """n x 3 (r, theta, phi) on the GPU and weights or None.  r from the selection times r^2 by the
    inverse of its cumulative distribution on a fine grid."""
    g = _gen(seed)
    u = torch.rand(3, n, dtype=torch.float64, device="cuda", generator=g)
    lo, hi = case["rmin"], case["rmax"]
    if case["window"] == "north":
        x = torch.linspace(lo, hi, 20001, dtype=torch.float64, device="cuda")
        d = _selection(case, x) * x * x
        c = torch.cat([torch.zeros(1, dtype=torch.float64, device="cuda"), torch.cumsum(0.5 * (d[1:] + d[:-1]), 0)])
        c = c / c[-1]
        i = torch.clamp(torch.searchsorted(c, u[0]), 1, x.numel() - 1)
        t = (u[0] - c[i - 1]) / (c[i] - c[i - 1])
        r = x[i - 1] + t * (x[i] - x[i - 1])
        cth = u[1]
    else:
        r = (u[0] * (hi ** 3 - lo ** 3) + lo ** 3) ** (1.0 / 3.0)
        cth = 1.0 - 2.0 * u[1]
    rtp = torch.stack([torch.clamp(r, lo, hi), torch.acos(cth), 2 * math.pi * u[2]], 1).contiguous()
    w = None
    if case["weights"]:
        w = (0.5 + torch.rand(n, dtype=torch.float32, device="cuda", generator=g)).double()
    return rtp, w


def _pix_theta(nside):
    """Colatitude of every ring-scheme pixel."""
    z, npr, _ = _rings(nside)
    return torch.repeat_interleave(torch.acos(z), npr)


def _mask(case, seed):
    npix = 12 * case["nside"] ** 2
    if case["window"] == "north":
        return (_pix_theta(case["nside"]) < 0.5 * math.pi).double().cuda()
    if case["window"] == "mask":  # a completeness map
        return 0.6 + 0.4 * torch.rand(npix, dtype=torch.float64, device="cuda", generator=_gen(seed + 5))
    return torch.ones(npix, dtype=torch.float64, device="cuda")


def _nbar(case, n):
    return n / (4 * math.pi / 3 * (case["rmax"] ** 3 - case["rmin"] ** 3)) * (2.0 if case["window"] == "north" else 1.0)


def _window(case, plan, seed):
    """(kind, a, b): device arrays of the window in the layout the transform takes."""
    am = plan.amodes
    wm = S.ConfigurationSpaceModes(case["rmin"], case["rmax"], 1000 if case["window"] != "dense" else 64, case["nside"])
    if case["window"] == "dense":
        th = _pix_theta(case["nside"]).numpy()
        x = (wm.r - wm.rmin) / (wm.rmax - wm.rmin)
        win = 0.5 + 0.4 * np.cos(th)[None, :] * x[:, None] + 0.1 * np.sin(3 * th)[None, :]
        W = plan.win_rhat_ln(win, wm)
        return L.SFB_WIN_DENSE, torch.from_numpy(np.nan_to_num(W.reshape(-1, order="F"))).cuda(), None
    phi = _selection(case, torch.from_numpy(wm.r)).numpy()
    w = plan.win_rhat_ln(S.SeparableArray(phi, np.ones(12 * am.nside ** 2)), wm)
    return L.SFB_WIN_SEPARABLE, _mask(case, seed), torch.from_numpy(w.arr2.reshape(-1, order="F").copy()).cuda()


def _cotangent(nlm, seed):
    return torch.randn(2 * nlm, dtype=torch.float64, device="cuda", generator=_gen(seed + 9))


def _field(case, seed):
    """A smooth field of nr shells plus noise, nr x npix column-major: [npix][nr] in memory."""
    npix = 12 * case["nside"] ** 2
    return torch.randn(npix, case["nr"], dtype=torch.float64, device="cuda", generator=_gen(seed + 3))


def _shells(case):
    wm = S.ConfigurationSpaceModes(case["rmin"], case["rmax"], case["nr"], case["nside"])
    return torch.from_numpy(np.ascontiguousarray(wm.r)).cuda(), float(wm.dr)


def prepare(case, seed):
    am = _modes(case)
    plan = S.Plan(am, precision=case["precision"])
    st = {"case": case, "plan": plan, "single": case["precision"] != "fp64"}
    nlm, kind = plan.nlmsize, case["kind"]
    if kind in ("cat", "mocks"):
        wk, wa, wb = _window(case, plan, seed)
        sizes = _sizes(case, seed)
        parts = [_catalogue(case, n, seed + 1000 * b) for b, n in enumerate(sizes)]
        st["nbar"] = [_nbar(case, n) for n in sizes]
        st["N"] = sizes
        if case["host"]:
            st["rtp"] = np.asfortranarray(parts[0][0].cpu().numpy().T)
            st["w"] = None if parts[0][1] is None else parts[0][1].cpu().numpy()
            if wk == L.SFB_WIN_DENSE:
                st["win"] = wa.cpu().numpy().reshape(plan.npix, am.lmax + 1, am.nmax, order="F")
            else:
                st["win"] = S.SeparableArray(wa.cpu().numpy(), wb.cpu().numpy().reshape(am.lmax + 1, am.nmax, order="F"),
                                             "mask", "w_ln")
        else:
            st["rtp"] = torch.cat([p[0] for p in parts])
            st["w"] = torch.cat([p[1] for p in parts]) if case["weights"] else None
            st["win"] = (wk, wa, wb)
            st["out"] = torch.empty(len(sizes) * 2 * nlm, dtype=torch.float64, device="cuda")
    elif kind == "vjp":
        st["rtp"], st["w"] = _catalogue(case, case["N"], seed)
        st["nbar"] = _nbar(case, case["N"])
        st["cot"] = _cotangent(nlm, seed)
        st["dr"] = torch.empty(case["N"], dtype=torch.float64, device="cuda")
        st["dw"] = torch.empty(case["N"], dtype=torch.float64, device="cuda")
    else:
        st["r"], st["delr"] = _shells(case)
        if kind == "field":
            st["in"] = _field(case, seed)
            st["out"] = torch.empty(2 * nlm, dtype=torch.float64, device="cuda")
        else:
            st["in"] = _cotangent(nlm, seed)
            st["out"] = torch.empty(plan.npix, case["nr"], dtype=torch.float64, device="cuda")
    return st


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def run(st):
    case, plan = st["case"], st["plan"]
    kind = case["kind"]
    if kind == "cat" and case["host"]:
        a = plan.cat2amln(st["rtp"], st["nbar"][0], st["win"], st["w"])
        return a.astype(np.complex64) if st["single"] else a
    if kind == "cat":
        plan.cat2amln_device(st["N"][0], st["rtp"], st["w"], st["nbar"][0], *st["win"], st["out"])
        return st["out"].float() if st["single"] else st["out"]
    if kind == "mocks":
        plan.cat2amln_batch_device(len(st["N"]), st["N"], st["rtp"], st["w"], st["nbar"], *st["win"], st["out"])
        return st["out"].float() if st["single"] else st["out"]
    if kind == "vjp":
        plan.cat2amln_vjp_device(case["N"], st["rtp"], st["w"], st["nbar"], st["cot"], st["dr"], st["dw"])
        return (st["dr"].float(), st["dw"].float()) if st["single"] else (st["dr"], st["dw"])
    fn = L.lib().sfb_field2anlm_device if kind == "field" else L.lib().sfb_anlm2field_device
    if kind == "field":
        L.check(fn(plan.handle, case["nr"], _ptr(st["r"]), st["delr"], _ptr(st["in"]), _ptr(st["out"]), None))
    else:
        L.check(fn(plan.handle, case["nr"], _ptr(st["r"]), _ptr(st["in"]), _ptr(st["out"]), None))
    return st["out"]


def work(case):
    """Inputs read once, outputs written once; the Legendre sum of every coefficient over the
    2 nside ring pairs (4 flop per complex term)."""
    am = _modes(case)
    npix, nlm = 12 * case["nside"] ** 2, S.getnlmsize(am)
    if case["kind"] in ("cat", "mocks"):
        n = case["N"] * case["mocks"]
        win = 8 * npix * am.nmaps if case["window"] == "dense" else 8 * (npix + am.nmaps)
        b = n * (24 + (8 if case["weights"] else 0)) + win + 16 * nlm * case["mocks"]
    elif case["kind"] == "vjp":
        b = case["N"] * (24 + 16 + (8 if case["weights"] else 0)) + 16 * nlm
    else:
        b = 8 * npix * case["nr"] + 16 * nlm
    return {"bytes": b, "flops": 4.0 * nlm * 2 * case["nside"] * case["mocks"]}


# ---- the same results in 64 bits with plain torch -----------------------------------------
# The radial spline tables (knots, values, second derivatives) are an input of the transform;
# everything from them on is written out here.


def _rings(nside):
    """cos(theta), pixel count and phi of the first pixel of the 4 nside - 1 rings."""
    i = torch.arange(1, 4 * nside, dtype=torch.float64)
    j = torch.minimum(i, 4 * nside - i)
    polar = j < nside
    z = torch.where(polar, 1 - j * j / (3.0 * nside * nside), (2 * nside - j) * 2.0 / (3.0 * nside))
    z = torch.where(i > 2 * nside, -z, z)
    npr = torch.where(polar, 4 * j, torch.full_like(j, 4 * nside)).long()
    shifted = polar | ((j - nside).long() % 2 == 0)
    phi0 = torch.where(shifted, math.pi / npr.double(), torch.zeros_like(z))
    return z, npr, phi0


def _ang2pix(nside, th, ph):
    z = torch.cos(th)
    za = z.abs()
    tt = torch.remainder(ph, 2 * math.pi) / (0.5 * math.pi)
    a, b = nside * (0.5 + tt), nside * z * 0.75
    jp, jm = torch.floor(a - b), torch.floor(a + b)
    ir = nside + 1 + jp - jm
    kshift = 1 - torch.remainder(ir, 2)
    ip = torch.remainder(torch.floor((jp + jm - nside + kshift + 1) / 2), 4 * nside)
    peq = 2 * nside * (nside - 1) + (ir - 1) * 4 * nside + ip
    tp = tt - torch.floor(tt)
    s = nside * torch.sqrt(3 * (1 - za))
    kp, km = torch.floor(tp * s), torch.floor((1 - tp) * s)
    ir = kp + km + 1
    ip = torch.remainder(torch.floor(tt * ir), 4 * ir)
    pn = 2 * ir * (ir - 1) + ip
    ps = 12 * nside * nside - 2 * ir * (ir + 1) + ip
    return torch.where(za <= 2.0 / 3.0, peq, torch.where(z > 0, pn, ps)).long()


class _SHT:
    """Ring analysis / synthesis of real maps [n][npix] as dense products, for m <= lmax."""

    def __init__(self, nside, lmax):
        self.nside, self.L, self.npix = nside, lmax, 12 * nside * nside
        self.dom = 4 * math.pi / self.npix
        z, npr, phi0 = _rings(nside)
        self.npr, self.phi0 = npr.tolist(), phi0.tolist()
        self.start = [0] + torch.cumsum(npr, 0).tolist()
        z = z.cuda()
        st = torch.sqrt((1 - z) * (1 + z))
        M = lmax + 1
        lam = torch.zeros(M, M, z.numel(), dtype=torch.float64, device="cuda")  # [l][m][ring]
        m = torch.arange(M, dtype=torch.float64, device="cuda")
        lognorm = torch.zeros(M, dtype=torch.float64, device="cuda")
        if lmax:
            k = torch.arange(1, M, dtype=torch.float64, device="cuda")
            lognorm[1:] = 0.5 * torch.cumsum(torch.log((2 * k + 1) / (2 * k)), 0)
        sign = 1 - 2 * torch.remainder(m, 2)
        diag = sign[:, None] * torch.exp(lognorm[:, None] + m[:, None] * torch.log(st)[None, :]) / math.sqrt(4 * math.pi)
        for l in range(M):
            lam[l, l] = diag[l]
            if l:
                mm = m[:l, None]
                a = torch.sqrt((4.0 * l * l - 1) / (l * l - mm * mm))
                prev = torch.sqrt(((l - 1.0) ** 2 - mm * mm).clamp(min=0) / (4 * (l - 1.0) ** 2 - 1)) if l > 1 else torch.zeros_like(mm)
                lam[l, :l] = a * (z[None, :] * lam[l - 1, :l] - (prev * lam[l - 2, :l] if l > 1 else 0.0))
        self.lam_mkl = lam.permute(1, 2, 0).contiguous()  # [m][ring][l]

    def _basis(self, ring):
        n = self.npr[ring]
        j = torch.arange(n, device="cuda")
        m = torch.arange(self.L + 1, device="cuda")
        ph = torch.remainder(j[:, None] * m[None, :], n).double() * (2 * math.pi / n) + self.phi0[ring] * m[None, :].double()
        return torch.cat([torch.cos(ph), -torch.sin(ph)], 1)  # [npr][2 M]: e^{-i m phi}

    def _runs(self):
        """Rings that share a basis: (first-pixel offsets, ring numbers)."""
        by = {}
        for k, (n, p) in enumerate(zip(self.npr, self.phi0)):
            by.setdefault((n, p), []).append(k)
        return by.values()

    def analysis(self, maps):
        """a[m][l][2 n] (re block, then im block)."""
        n, M = maps.shape[0], self.L + 1
        F = torch.empty(M, len(self.npr), 2 * n, dtype=torch.float64, device="cuda")
        for run in self._runs():
            B, c = self._basis(run[0]), self.npr[run[0]]
            x = torch.stack([maps[:, self.start[k]:self.start[k] + c] for k in run])
            y = (x.reshape(-1, c) @ B).reshape(len(run), n, 2, M)
            F[:, run] = y.permute(3, 0, 2, 1).reshape(M, len(run), 2 * n)
        return self.dom * torch.bmm(self.lam_mkl.transpose(1, 2).contiguous(), F)

    def synthesis(self, a):
        n, M = a.shape[2] // 2, self.L + 1
        G = torch.bmm(self.lam_mkl, a)  # [m][ring][2 n]
        G[1:] *= 2.0
        out = torch.empty(n, self.npix, dtype=torch.float64, device="cuda")
        for run in self._runs():
            B, c = self._basis(run[0]), self.npr[run[0]]
            g = G[:, run].reshape(M, len(run), 2, n).permute(1, 3, 2, 0).reshape(-1, 2 * M)
            y = (g @ B.T.contiguous()).reshape(len(run), n, c)
            for i, k in enumerate(run):
                out[:, self.start[k]:self.start[k] + c] = y[i]
        return out

    def map2alm(self, maps, niter=3):
        a = self.analysis(maps)
        for _ in range(niter):
            a = a + self.analysis(maps - self.synthesis(a))
        return a

    def refine(self, b, niter=3):
        """sum_{j <= niter} (1 - A S)^j b."""
        a = b
        for _ in range(niter):
            a = b + a - self.analysis(self.synthesis(a))
        return a


def _splines(am, q):
    o0, o1 = int(am.knot_off[q]), int(am.knot_off[q + 1])
    return tuple(torch.from_numpy(np.ascontiguousarray(v[o0:o1])).cuda() for v in (am.knot_x, am.knot_y, am.knot_ypp))


class _Radial:
    """Spline values and slopes of map after map at fixed radii (knots shared by runs of maps)."""

    def __init__(self, am, r):
        self.am, self.r, self.cache = am, r, {}

    def __call__(self, q, slope=False):
        x, y, ypp = _splines(self.am, q)
        n = x.numel()
        seg = self.cache.get(n)
        if seg is None or not torch.equal(seg[0], x):
            i = torch.clamp(torch.searchsorted(x, self.r, right=True) - 1, 0, n - 2)
            h = x[1:] - x[:-1]
            u = ((self.r - x[i]) / h[i]).clamp(0.0, 1.0)
            seg = self.cache[n] = (x, i, u, h)
        _, i, u, h = seg
        c = torch.stack([y[:-1], y[1:] - y[:-1] - h * h * (2 * ypp[:-1] + ypp[1:]) / 6, h * h * ypp[:-1] / 2,
                         h * h * (ypp[1:] - ypp[:-1]) / 6], 1)[i]
        g = c[:, 0] + u * (c[:, 1] + u * (c[:, 2] + u * c[:, 3]))
        if not slope:
            return g
        return g, (c[:, 1] + u * (2 * c[:, 2] + 3 * u * c[:, 3])) / h[i]


def _maps_of(am):
    return [(n, l) for n in range(1, am.nmax + 1) for l in range(int(am.lmax_n[n - 1]) + 1)]


def _pack(am, qs, a, out, base):
    """Rows l of the maps qs from a[m][l][2 n] to the interleaved a_nlm vector."""
    n = len(qs)
    for i, (q, l) in enumerate(qs):
        o = base[q]
        out[o:o + 2 * (l + 1):2] = a[:l + 1, l, i]
        out[o + 1:o + 2 * (l + 1):2] = a[:l + 1, l, n + i]


def _bases(maps):
    base, o = [], 0
    for _, l in maps:
        base.append(o)
        o += 2 * (l + 1)
    return base, o


def _interleave(path_real, complex_out):
    if not complex_out:
        return path_real
    return torch.view_as_complex(path_real.reshape(-1, 2).contiguous()).cpu().numpy()


def exact(case, seed):
    am = _modes(case)
    maps = _maps_of(am)
    base, size = _bases(maps)
    sht = _SHT(case["nside"], am.lmax)
    chunk = max(1, min(len(maps), int(3e8 // sht.npix)))
    kind = case["kind"]
    if kind in ("cat", "mocks"):
        plan = S.Plan(am, precision="fp64")
        wk, wa, wb = _window(case, plan, seed)
        plan.close()
        res = []
        for b, n in enumerate(_sizes(case, seed)):
            rtp, w = _catalogue(case, n, seed + 1000 * b)
            pix, rad = _ang2pix(case["nside"], rtp[:, 1], rtp[:, 2]), _Radial(am, rtp[:, 0].contiguous())
            inv = 1.0 / (_nbar(case, n) * sht.dom)
            out = torch.empty(size, dtype=torch.float64, device="cuda")
            for q0 in range(0, len(maps), chunk):
                qs = list(range(q0, min(q0 + chunk, len(maps))))
                d = torch.zeros(len(qs), sht.npix, dtype=torch.float64, device="cuda")
                for i, q in enumerate(qs):
                    g = rad(q)
                    d[i].index_add_(0, pix, g if w is None else g * w)
                    at = maps[q][1] + (am.lmax + 1) * (maps[q][0] - 1)
                    W = wa[at * sht.npix:(at + 1) * sht.npix] if wk == L.SFB_WIN_DENSE else wa * wb[at]
                    d[i] = d[i] * inv - W
                _pack(am, [(q, maps[q][1]) for q in qs], sht.map2alm(d), out, base)
            res.append(out)
        return _interleave(torch.cat(res), case["host"])
    if kind == "vjp":
        rtp, w = _catalogue(case, case["N"], seed)
        pix, rad = _ang2pix(case["nside"], rtp[:, 1], rtp[:, 2]), _Radial(am, rtp[:, 0].contiguous())
        cot = _cotangent(size // 2, seed)
        dr, dw = torch.zeros_like(rtp[:, 0]), torch.zeros_like(rtp[:, 0])
        M = am.lmax + 1
        for q0 in range(0, len(maps), chunk):
            qs = list(range(q0, min(q0 + chunk, len(maps))))
            c = torch.zeros(M, M, 2 * len(qs), dtype=torch.float64, device="cuda")
            for i, q in enumerate(qs):
                l, o = maps[q][1], base[q]
                c[:l + 1, l, i] = cot[o:o + 2 * (l + 1):2]
                c[:l + 1, l, len(qs) + i] = cot[o + 1:o + 2 * (l + 1):2]
            c[1:] *= 0.5
            c[0, :, len(qs):] = 0.0
            bar = sht.synthesis(sht.refine(c)) * sht.dom
            for i, q in enumerate(qs):
                g, gp = rad(q, slope=True)
                v = bar[i][pix]
                dw += g * v
                dr += gp * v
        inv = 1.0 / (_nbar(case, case["N"]) * sht.dom)
        return dr * inv if w is None else dr * inv * w, dw * inv
    r, delr = _shells(case)
    rad = _Radial(am, r)
    G = torch.stack([rad(q) for q in range(len(maps))])  # [map][nr]
    if kind == "field":
        a = sht.map2alm(_field(case, seed).T.contiguous())  # [m][l][2 nr]
        nr, out = case["nr"], torch.empty(size, dtype=torch.float64, device="cuda")
        c = G * (delr * r * r)
        for q, (_, l) in enumerate(maps):
            v = a[:l + 1, l].reshape(l + 1, 2, nr) @ c[q]
            out[base[q]:base[q] + 2 * (l + 1)] = v.reshape(-1)
        return out
    cot = _cotangent(size // 2, seed)
    a = torch.zeros(am.lmax + 1, am.lmax + 1, 2, case["nr"], dtype=torch.float64, device="cuda")
    for q, (_, l) in enumerate(maps):
        a[:l + 1, l] += cot[base[q]:base[q] + 2 * (l + 1)].reshape(l + 1, 2)[:, :, None] * G[q]
    a[0, :, 1] = 0.0  # a real field: the m = 0 coefficients enter with their real parts
    return sht.synthesis(a.reshape(am.lmax + 1, am.lmax + 1, -1)).T.contiguous()
