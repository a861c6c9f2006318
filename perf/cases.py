"""The work users of this framework have it do, as cases to be timed.

Each case is one stage of a run_tile / run_multitile_split tile, called through
the package as a program calls it, with the mesh sizes and filter banks of
``pipeline.CONFIGS`` and the serving stream (``serve.SERVE_*``):

  fields   the input fields of a periodic tile (run_tile)
  split    the fields of one tile of a multi-resolution run
  coarse   the coarse fields of such a run, made once per run
  peaks    filter bank and peak stencil
  shell    radial-shell analysis of a tile's peaks
  tile     peaks -> bookkeeping -> shell analysis -> halo records in one go
  merge    exclusion and volume reduction of a halo catalogue

``listed`` names the cases, ``draw`` gives further ones of the same ranges,
``prepare`` makes a case's inputs from a seed with torch, ``run`` is one pass,
``work`` what a pass cannot do without, ``exact`` its outputs in 64 bits.

Lists whose length depends on the field (peaks, records, merged halos) are
handed on in buffers of a fixed number of rows, as a program with static
shapes keeps them: the rows past the end hold zeros.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "peakpatch.jl_amd"))

from peakpatch_hip import SHELL_PERSISTENT, Context, catalog, collapse, split, synth  # noqa: E402
from peakpatch_hip.api import PeakList  # noqa: E402
from peakpatch_hip.pipeline import TileConfig, TileDriver  # noqa: E402

ALATT = 250.0 / 256.0  # Mpc/h, the cell of the 256^3 and of the served tiles


def listed():
    c1 = dict(n=128, alatt=75.0 / 128, nfilt=10, rf_min=1.5, rf_max=8.0, lightcone=False, z=0.0)
    c2 = dict(alatt=ALATT, nfilt=20, rf_min=1.0, rf_max=15.0)
    c3 = dict(n=512, alatt=600.0 / 512, nfilt=25, rf_min=1.0, rf_max=30.0, lightcone=True, z=4.6)
    return [
        # the smallest run: a 128^3 box, first-order displacements, no shear output
        dict(name="fields_128", kind="fields", n=128, alatt=75.0 / 128, ilpt=1, lapd=False),
        # a mesh that is no power of two, second order and the k^2 field
        dict(name="fields_250", kind="fields", n=250, alatt=ALATT, ilpt=2, lapd=True),
        # the 512^3 light-cone tile's inputs
        dict(name="fields_512", kind="fields", n=512, alatt=600.0 / 512, ilpt=2, lapd=True),
        # tiles of multi-resolution runs: a small one and a large one of the serving stream's kind
        dict(name="split_192", kind="split", n=192, alatt=ALATT, ntile=4, nbuff=27, ilpt=2, lapd=True),
        dict(name="split_512", kind="split", n=512, alatt=ALATT, ntile=4, nbuff=27, ilpt=2, lapd=True),
        # the coarse fields every tile of a 256^3-tile run shares
        dict(name="coarse_256", kind="coarse", n=256, alatt=ALATT, ntile=4, nbuff=27),
        # filter bank and stencil: the smallest configuration, host arrays out; the light-cone tile, left on the device
        dict(name="peaks_128", kind="peaks", lapd=False, device_out=False, **c1),
        dict(name="peaks_512", kind="peaks", lapd=True, device_out=True, **c3),
        # shell analysis of the same two tiles: two thousand peaks, two million
        dict(name="shell_128", kind="shell", npeaks=2000, ilpt=1, lapd=False, **c1),
        dict(name="shell_512", kind="shell", npeaks=1950000, ilpt=2, lapd=True, **c3),
        # one served light-cone tile of a ragged size from its fields to its records
        dict(name="tile_200", kind="tile", n=200, lightcone=True, z=4.6, **c2),
        # the merge of a run's catalogue
        dict(name="merge_1200007", kind="merge", n=1200007, box=600.0, extended=True),
    ]


def _mesh(rng, lo, hi):
    """A mesh size in [lo, hi], spread over its logarithm: mostly even with
    factors up to 7, as meshes are chosen for their transforms, one in four any."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.25:
        return n

    def smooth(v):
        for p in (2, 3, 5, 7):
            while v % p == 0:
                v //= p
        return v == 1
    return min((m for m in range(lo, hi + 1) if m % 2 == 0 and smooth(m)), key=lambda m: (abs(m - n), m))


def draw(rng):
    kind = rng.choice(("fields", "split", "coarse", "peaks", "shell", "tile", "merge"))
    alatt = round(rng.uniform(0.45, 1.2), 4)
    if kind == "merge":
        n = int(round(math.exp(rng.uniform(math.log(300), math.log(1.2e6)))))
        return dict(kind=kind, n=n, box=round(max(40.0, 600.0 * (n / 1.2e6) ** (1 / 3)), 2), extended=rng.random() < 0.5)
    if kind == "fields":
        ilpt = rng.choice((1, 2, 2))
        return dict(kind=kind, n=_mesh(rng, 32, 480), alatt=alatt, ilpt=ilpt, lapd=rng.random() < 0.7)
    if kind in ("split", "coarse"):
        n = _mesh(rng, 64, 448 if kind == "split" else 256)
        c = dict(kind=kind, n=n, alatt=alatt, ntile=rng.choice((2, 3, 4)), nbuff=rng.randint(4, n // 8))
        return c if kind == "coarse" else dict(c, ilpt=rng.choice((1, 2, 2)), lapd=rng.random() < 0.7)
    n = _mesh(rng, 48, {"peaks": 400, "shell": 300, "tile": 288}[kind])
    rf_min = alatt * rng.uniform(0.9, 2.6)
    cone = rng.random() < 0.5
    c = dict(kind=kind, n=n, alatt=alatt, nfilt=rng.randint(3, 20), rf_min=round(rf_min, 3),
             rf_max=round(max(1.5 * rf_min, alatt * n * rng.uniform(0.05, 0.11)), 3), lightcone=cone,
             z=4.6 if cone else round(rng.uniform(0.0, 1.0), 2))
    if kind == "peaks":
        return dict(c, lapd=rng.random() < 0.7, device_out=rng.random() < 0.5)
    if kind == "tile":
        return c
    npeaks = max(50, int(_inner(c) * 0.012 * (0.9 * alatt / rf_min) ** 3))
    return dict(c, npeaks=npeaks, ilpt=rng.choice((1, 2, 2)), lapd=rng.random() < 0.7)


def _inner(case):
    """Cells of the cube the stencil searches."""
    return max(0, case["n"] - 2 * (int(1.75 * case["rf_max"] / case["alatt"]) + 1)) ** 3


def _capacity(case):
    """Rows of the buffers for the peaks or records of a tile: a filtered
    field has under one maximum in thirty cells."""
    return _inner(case) // 30 + 64


# ------------------------------------------------------------------ inputs
_CTX = {}
_PEAK = ("i", "j", "k", "filt", "delta_s", "lapd_s")


def _context(case):
    """The context a program holds for its run: one for the stages without
    shell tables, one per shell radius with them and the collapse table."""
    rmax = _config(case).nhunt if case["kind"] in ("shell", "tile") else None
    if rmax not in _CTX:
        ctx = _CTX[rmax] = Context(0)
        if rmax is not None:
            ct = collapse.read_homeltab(os.path.join("tests", "golden", "HomelTab_fortran.dat"))
            ctx.upload_collapse_table(ct.table, *ct.bounds)
            ctx.build_shell_tables(rmax)
    return _CTX[rmax]


def _config(case):
    n, box = case["n"], case["n"] * case["alatt"]
    full = case["kind"] == "tile"
    cone = case["lightcone"]
    return TileConfig("case", n, box, case["nfilt"], case["rf_min"], case["rf_max"],
                      ilpt=2 if full else case.get("ilpt", 1), ioutshear=1 if full or case["lapd"] else 0,
                      ievol=1 if cone else 0, z_out=0.0 if cone else case["z"], z_max=case["z"] if cone else 0.0,
                      cen=(-box / 2,) * 3 if cone else (0.0,) * 3)


def _geometry(case, seed):
    return split.geometry(case["n"], case["nbuff"], case["ntile"], case["alatt"], seed=seed)


def _power(k):
    """Eisenstein & Hu (1998) no-wiggle P(k) / (2 pi)^3 of the configurations'
    cosmology, sigma_8 = 0.808 (numpy, Float64)."""
    Om, Ob, h, ns, s8 = 0.315, 0.049, 0.674, 0.965, 0.808
    om, ob, fb, th = Om * h * h, Ob * h * h, Ob / Om, 2.7255 / 2.7
    s = 44.5 * math.log(9.83 / om) / math.sqrt(1 + 10 * ob ** 0.75)
    al = 1 - 0.328 * math.log(431 * om) * fb + 0.38 * math.log(22.3 * om) * fb * fb

    def p(k):
        q = k * th ** 2 / (Om * h * (al + (1 - al) / (1 + (0.43 * k * h * s) ** 4)))
        L = np.log(2 * math.e + 1.8 * q)
        return k ** ns * (L / (L + (14.2 + 731 / (1 + 62.5 * q)) * q * q)) ** 2
    lk = np.linspace(math.log(1e-5), math.log(1e3), 20001)
    kk = np.exp(lk)
    x = kk * 8.0
    with np.errstate(invalid="ignore"):
        w = np.where(x > 1e-4, 3 * (np.sin(x) - x * np.cos(x)) / x ** 3, 1 - x * x / 10)
    f = kk ** 3 * p(kk) * w * w / (2 * math.pi ** 2)
    var = float(np.sum((f[1:] + f[:-1]) / 2 * np.diff(lk)))
    return p(k) * s8 * s8 / var / (2 * math.pi) ** 3


_TABLE = []


def _power_at(k):
    """P of a Float64 tensor of k > 0 through the log-log table programs read:
    2001 rows from 1e-4 to 1e2 h/Mpc, extrapolated linearly."""
    if not _TABLE:
        lk = np.linspace(math.log(1e-4), math.log(1e2), 2001)
        tk = np.exp(lk)
        _TABLE.append([torch.as_tensor(np.log(v), device="cuda") for v in (tk, _power(tk))])
    lk, lp = _TABLE[0]
    x = torch.log(k)
    i = (torch.searchsorted(lk, x.contiguous(), right=True) - 1).clamp_(0, len(lk) - 2)
    return torch.exp(lp[i] + (x - lk[i]) / (lk[i + 1] - lk[i]) * (lp[i + 1] - lp[i]))


def _waves(n, box, dtype):
    """kx, ky, kz (broadcastable) of the half spectrum; the Nyquist index of
    the full axes is the negative frequency."""
    f = torch.arange(n, device="cuda")
    f = torch.where(f < (n + 1) // 2, f, f - n).to(torch.float64) * (2 * math.pi / box)
    x = torch.arange(n // 2 + 1, device="cuda").to(torch.float64) * (2 * math.pi / box)
    return x[None, None, :].to(dtype), f[None, :, None].to(dtype), f[:, None, None].to(dtype)


def _irfftn(a, n):
    """Normalised inverse of a half spectrum: the imaginary parts left on the
    kx = 0 and Nyquist planes after the two full axes are dropped."""
    a = torch.fft.ifft(torch.fft.ifft(a, dim=0), dim=1)
    a[:, :, 0].imag.zero_()
    if n % 2 == 0:
        a[:, :, -1].imag.zero_()
    return torch.fft.irfft(a, n=n, dim=2)


def _delta(case, seed):
    """A Gaussian density field of the configurations' power spectrum."""
    n, box = case["n"], case["n"] * case["alatt"]
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    dk = torch.fft.rfftn(torch.randn((n, n, n), generator=g, device="cuda"))
    kx, ky, kz = _waves(n, box, torch.float64)
    for q in range(n):  # plane by plane: the Float64 temporaries stay small
        k2 = kx[0] ** 2 + ky[0] ** 2 + kz[q] ** 2
        if q == 0:
            k2[0, 0] = 1.0
        dk[q] *= torch.sqrt(_power_at(torch.sqrt(k2)) * (2 * math.pi / box) ** 3 * float(n) ** 3).to(torch.float32)
    dk[0, 0, 0] = 0
    return torch.fft.irfftn(dk, s=(n, n, n)).contiguous()


def _displacements(delta, box, ilpt, lapd):
    """(eta, eta2, lapd) of a density field, Float32."""
    n = delta.shape[0]
    dk = torch.fft.rfftn(delta)
    k = _waves(n, box, torch.float32)
    k2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    lap = torch.fft.irfftn(dk * k2, s=(n, n, n)) / float(n) ** 3 if lapd else None
    k2[0, 0, 0] = 1.0

    def grad(a, sign):
        a[0, 0, 0] = 0
        if n % 2 == 0:
            a[:, :, -1] = 0
            a[:, n // 2] = 0
            a[n // 2] = 0
        return tuple(torch.fft.irfftn(a * (sign * 1j * k[q]), s=(n, n, n)) for q in range(3))
    eta2 = None
    if ilpt >= 2:
        p = {ab: torch.fft.irfftn(dk * (-k[ab[0]] * k[ab[1]] / k2), s=(n, n, n))
             for ab in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))}
        src = sum(p[a, a] * p[b, b] - p[a, b] ** 2 for a, b in ((0, 1), (0, 2), (1, 2)))
        del p
        eta2 = grad(torch.fft.rfftn(src) / k2, -1)
    return grad(dk / k2, 1), eta2, lap


def _windows(n, box, Rf, dtype):
    """(top-hat, k^2-Gaussian) windows of one filter, evaluated in Float64."""
    kx, ky, kz = _waves(n, box, torch.float64)
    k = torch.sqrt(kx ** 2 + ky ** 2 + kz ** 2)
    x = k * Rf
    x[0, 0, 0] = 1.0
    top = 3 * (torch.sin(x) - x * torch.cos(x)) / x ** 3
    top[0, 0, 0] = 1.0
    gauss = k * k * torch.exp(-(k * Rf) ** 2 / 8)
    gauss[0, 0, 0] = 1.0
    return top.to(dtype), gauss.to(dtype)


def _find(delta, case, fcrit, lapd):
    """Filter bank and stencil in torch, in delta's precision: the peaks of
    every filter in (k, j, i) order, a cell at most once."""
    n, box = case["n"], case["n"] * case["alatt"]
    cfg = _config(case)
    b = cfg.nbuff_eff
    dk = torch.fft.rfftn(delta)
    free = torch.zeros((n, n, n), dtype=torch.bool, device="cuda")
    free[b:n - b, b:n - b, b:n - b] = True
    rows = []
    for f, Rf in enumerate(cfg.filters):
        top, gauss = _windows(n, box, float(Rf), delta.dtype)
        s = torch.fft.irfftn(dk * top, s=(n, n, n))
        m = s
        for d in range(3):
            m = torch.maximum(torch.maximum(m, m.roll(1, d)), m.roll(-1, d))
        cells = torch.nonzero((s >= m) & (s >= float(fcrit[f])) & free)
        at = tuple(cells.T)
        free[at] = False
        i32 = cells.to(torch.int32)
        rows.append((i32[:, 2], i32[:, 1], i32[:, 0], torch.full_like(i32[:, 0], f), s[at],
                     torch.fft.irfftn(dk * gauss, s=(n, n, n))[at] if lapd else None))
    cat = [torch.cat([r[q] for r in rows]).contiguous() if rows[0][q] is not None else None for q in range(6)]
    return PeakList(*cat)


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case, seed=int(seed), ctx=_context(case))
    if kind in ("split", "coarse"):
        s["geom"] = _geometry(case, s["seed"])
        if kind == "split":
            s["coarse"] = split.CoarseField(s["ctx"], s["geom"])
            s["tile"] = tuple(1 + (s["seed"] // case["ntile"] ** q) % case["ntile"] for q in range(3))
    elif kind == "merge":
        s["records"] = _catalogue(case, s["seed"])
    elif kind in ("peaks", "shell", "tile"):
        cfg = _config(case)
        s["driver"] = drv = TileDriver(cfg)
        s["delta"] = _delta(case, s["seed"])
        if kind != "peaks":
            s["fields"] = (s["delta"], *_displacements(s["delta"], cfg.boxsize, cfg.ilpt, cfg.ioutshear >= 1))
        if kind == "shell":
            # a batch of a fixed number of peaks, evenly out of the tile's
            batch = drv.device_batch(s["ctx"], _find(s["delta"], case, drv.filter_fcrit(), cfg.ioutshear >= 1))
            rows = torch.arange(case["npeaks"], device="cuda") * len(batch["i"]) // case["npeaks"]
            s["batch"] = {k: v[rows] for k, v in batch.items()}
    return s


def _catalogue(case, seed):
    """Halo records as a run's shell analysis leaves them: centres clustered
    around common neighbours, many radii near the smallest filter's, few large."""
    n, box = case["n"], case["box"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: torch.rand(s, generator=g, device="cuda")  # noqa: E731
    nor = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    rec = torch.zeros((n, 33 if case["extended"] else 11), device="cuda")
    rec[:, 7:] = nor(n, rec.shape[1] - 7)
    parents = rnd(max(1, n // 6), 3) * box
    which = (rnd(n) * len(parents)).long().clamp_(max=len(parents) - 1)
    rec[:, :3] = parents[which] + 3.0 * nor(n, 3)
    rec[:, 3:6] = 5.0 * nor(n, 3)
    rec[:, 6] = torch.clamp(1.2 * (1.0 - rnd(n)) ** (-1 / 3.2), max=15.0)
    return rec


# --------------------------------------------------------------- one pass
def _rows(a, count):
    """a (a list of peaks or records) in a buffer of count rows."""
    if a is None:
        return None
    if len(a) > count:
        raise ValueError(f"{len(a)} rows in a buffer of {count}")
    out = a.new_zeros((count, *a.shape[1:])) if isinstance(a, torch.Tensor) else np.zeros((count, *a.shape[1:]), a.dtype)
    out[:len(a)] = a
    return out


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "fields":
        t = synth.make_tile(ctx, case["n"], case["n"] * case["alatt"], seed=s["seed"], ilpt=case["ilpt"],
                            want_lapd=case["lapd"])
        return dict(delta=t.delta, eta=t.eta, eta2=t.eta2, lapd=t.lapd)
    if kind == "split":
        t = split.make_split_tile(ctx, s["coarse"], *s["tile"], ilpt=case["ilpt"], want_lapd=case["lapd"])
        return dict(delta=t.delta, eta=t.eta, eta2=t.eta2, lapd=t.lapd)
    if kind == "coarse":
        c = split.CoarseField(ctx, s["geom"])
        noise, delta, psi = c.download()
        c.close()
        return dict(noise=noise, delta=delta, psi=psi)
    if kind == "merge":
        return _rows(catalog.merge_catalog(ctx, s["records"]), case["n"])
    drv = s["driver"]
    if kind == "peaks":
        p = drv.find_peaks(ctx, s["delta"], device_out=case["device_out"])
        return dict(count=len(p), **{f: _rows(getattr(p, f), _capacity(case)) for f in _PEAK})
    n = case["n"]
    mask = torch.zeros((n, n, n), dtype=torch.int8, device="cuda")
    if kind == "shell":
        r = drv.analyse(ctx, s["fields"], s["batch"], mask=mask, kernel=SHELL_PERSISTENT, device_out=True)
        return dict(r, mask=mask)
    peaks = drv.find_peaks(ctx, s["delta"], device_out=True)
    batch = drv.device_batch(ctx, peaks, round_f32=True)
    r = drv.analyse(ctx, s["fields"], batch, mask=mask, kernel=SHELL_PERSISTENT, device_out=True)
    records, rmax = catalog.pack_halos(ctx, r, batch, case["alatt"], True)
    return dict(count=len(records), records=_rows(records, _capacity(case)), RTHLmax=rmax, mask=mask)


# -------------------------------------------------------------- the floor
def work(case):
    """Inputs read once and outputs written once; the transforms' operations
    (5 N log2 N per complex transform, half of it for real data), with peak
    counts of about 1.5 in a hundred cells."""
    kind, n3 = case["kind"], float(case["n"]) ** 3
    fft = lambda m: 2.5 * m * math.log2(max(m, 2.0))  # noqa: E731
    if kind == "merge":
        return dict(bytes=2.0 * case["n"] * 4 * (33 if case["extended"] else 11), flops=0.0)
    if kind in ("fields", "split"):
        outs = 4 + (3 if case["ilpt"] >= 2 else 0) + (1 if case["lapd"] else 0)
        pots = 7 if case["ilpt"] >= 2 else 0
        if kind == "fields":
            return dict(bytes=4.0 * n3 * outs, flops=(1 + outs + pots) * fft(n3))
        return dict(bytes=4.0 * n3 * outs, flops=5 * fft(8 * n3) + (outs - 3 + pots) * fft(n3))
    if kind == "coarse":
        g = _geometry(case, 0)
        return dict(bytes=20.0 * g.M ** 3, flops=100.0 * float(g.N) ** 3)  # a Threefry block and a normal per cell
    per = 0.015 * n3
    banks = (2 if case.get("lapd", True) else 1) * case["nfilt"]
    if kind == "peaks":
        return dict(bytes=4 * n3 + 24 * per, flops=(1 + banks) * fft(n3))
    fields = 8 if kind == "tile" else 4 + (3 if case["ilpt"] >= 2 else 0) + (1 if case["lapd"] else 0)
    if kind == "shell":
        return dict(bytes=(4 * fields + 1) * n3 + (56 + 248) * per, flops=30 * 400 * per)
    return dict(bytes=(4 * fields + 1) * n3 + 132 * per, flops=(1 + banks) * fft(n3) + 30 * 400 * per)


# ------------------------------------------------------------ in 64 bits
def _normals(pair, seed):
    """The two Float64 normals of Threefry-2x64-20 counters (pair, 0) under
    key (seed, 0), uniforms of 53 bits, Box-Muller (int64 tensors wrap)."""
    wrap = lambda v: (v + (1 << 63)) % (1 << 64) - (1 << 63)  # noqa: E731
    ks = [wrap(seed), 0, wrap(0x1BD11BDAA9FC1A22 ^ seed)]
    x0, x1 = pair + ks[0], torch.full_like(pair, ks[1])
    for b in range(5):
        for q in range(4):
            r = (16, 42, 12, 31, 16, 32, 24, 21)[(4 * b + q) % 8]
            x0 = x0 + x1
            x1 = ((x1 << r) | ((x1 >> (64 - r)) & ((1 << r) - 1))) ^ x0
        x0 = x0 + ks[(b + 1) % 3]
        x1 = x1 + wrap(ks[(b + 2) % 3] + b + 1)
    u = [(((x >> 11) & ((1 << 53) - 1)).to(torch.float64) + 1.0) * 2.0 ** -53 for x in (x0, x1)]
    r, t = torch.sqrt(-2.0 * torch.log(u[0])), 2 * math.pi * u[1]
    return r * torch.cos(t), r * torch.sin(t)


def _noise(idx, seed):
    """The normals of 0-based cell numbers, as the Float32 values fields hold."""
    a, b = _normals(idx >> 1, seed)
    return torch.where(idx % 2 == 0, a, b).to(torch.float32).to(torch.float64)


def _amplitude(k2, dk, n):
    z = k2 == 0
    a = torch.sqrt(_power_at(torch.sqrt(torch.where(z, torch.ones_like(k2), k2))) * dk ** 3 * float(n) ** 3)
    return torch.where(z, torch.zeros_like(a), a)


def _planes(spec, k, dk, factor):
    """spec with each kz plane times factor(k2, kx, ky, kz)."""
    out = torch.empty_like(spec)
    for q in range(spec.shape[0]):
        kz = k[2][q]
        out[q] = spec[q] * factor(k[0][0] ** 2 + k[1][0] ** 2 + kz ** 2, k[0][0], k[1][0], kz)
    return out


def _second(delta, box, ilpt, lapd, split_rules):
    """(eta2, k^2 field) of a density field in 64 bits, by run_tile's formulas
    or by the split tiles' (k = 0 and Nyquist zeroed throughout)."""
    n = delta.shape[0]
    k = _waves(n, box, torch.float64)
    nyq = torch.zeros((n, n, n // 2 + 1), dtype=torch.bool, device="cuda")
    nyq[:, :, n // 2] = True
    nyq[:, n // 2] = True
    nyq[n // 2] = True
    safe = lambda k2: torch.where(k2 == 0, torch.ones_like(k2), k2)  # noqa: E731
    dk = torch.fft.rfftn(delta)
    if split_rules:
        dk = dk.masked_fill(nyq, 0)
    dk[0, 0, 0] = 0
    lap = _irfftn(_planes(dk, k, 0, lambda k2, x, y, z: k2), n) / (1.0 if split_rules else float(n) ** 3) if lapd else None
    eta2 = None
    if ilpt >= 2:
        ax = lambda q, x, y, z: (x, y, z)[q]  # noqa: E731
        phi = lambda a, b: _irfftn(_planes(dk, k, 0, lambda k2, x, y, z: -ax(a, x, y, z) * ax(b, x, y, z) / safe(k2)), n)  # noqa: E731
        if split_rules:
            src = delta * delta / 2
            for q in range(3):
                src -= phi(q, q) ** 2 / 2
            for a, b in ((0, 1), (0, 2), (1, 2)):
                src -= phi(a, b) ** 2
        else:
            d = [phi(q, q) for q in range(3)]
            src = sum(d[a] * d[b] - phi(a, b) ** 2 for a, b in ((0, 1), (0, 2), (1, 2)))
        sk = torch.fft.rfftn(src).masked_fill(nyq, 0)
        sk[0, 0, 0] = 0
        eta2 = tuple(_irfftn(_planes(sk, k, 0, lambda k2, x, y, z: -1j * ax(q, x, y, z) / safe(k2)), n) for q in range(3))
    return eta2, lap


def _exact_fields(case, seed):
    n, box = case["n"], case["n"] * case["alatt"]
    dk = 2 * math.pi / box
    k = _waves(n, box, torch.float64)
    noise = torch.empty(n * n * n, dtype=torch.float64, device="cuda")
    for a in range(0, n ** 3, 1 << 24):
        noise[a:a + (1 << 24)] = _noise(torch.arange(a, min(n ** 3, a + (1 << 24)), device="cuda"), seed)
    spec = _planes(torch.fft.rfftn(noise.view(n, n, n)), k, dk, lambda k2, x, y, z: _amplitude(k2, dk, n))
    delta = _irfftn(spec.clone(), n)
    spec = torch.fft.rfftn(delta)
    spec[:, :, n // 2] = 0
    spec[:, n // 2] = 0
    spec[n // 2] = 0
    spec[0, 0, 0] = 0
    safe = lambda k2: torch.where(k2 == 0, torch.ones_like(k2), k2)  # noqa: E731
    eta = tuple(_irfftn(_planes(spec, k, dk, lambda k2, x, y, z: 1j * (x, y, z)[q] / safe(k2)), n) for q in range(3))
    eta2, lap = _second(delta, box, case["ilpt"], case["lapd"], False)
    return dict(delta=delta, eta=eta, eta2=eta2, lapd=lap)


def _exact_coarse(g):
    """(noise, delta, psi) of the coarse grid in 64 bits."""
    N, M, b = g.N, g.M, g.block
    noise = torch.empty((M, M, M), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 24) // (N * N))
    for K in range(M):
        acc = torch.zeros((M, M), dtype=torch.float64, device="cuda")
        for z in range(K * b, (K + 1) * b, step):
            m = min(step, (K + 1) * b - z)
            first, last = z * N * N, (z + m) * N * N
            a, c = _normals(torch.arange(first >> 1, (last + 1) >> 1, device="cuda"), g.seed)
            v = torch.stack((a, c), 1).view(-1)[first & 1:][:last - first]
            acc += v.view(m, M, b, M, b).sum((0, 2, 4))
        noise[K] = acc / math.sqrt(float(b) ** 3)
    box = N * g.alatt
    dk = 2 * math.pi / box
    k = _waves(M, box, torch.float64)
    spec = _planes(torch.fft.rfftn(noise), k, dk, lambda k2, x, y, z: _amplitude(k2, dk, M))
    safe = lambda k2: torch.where(k2 == 0, torch.ones_like(k2), k2)  # noqa: E731
    psi = tuple(_irfftn(_planes(spec, k, dk, lambda k2, x, y, z: 1j * (x, y, z)[q] / safe(k2)), M) for q in range(3))
    return noise, _irfftn(spec.clone(), M), psi


def _interpolated(coarse, g, tile):
    """Catmull-Rom interpolation of a coarse field onto the tile's cells."""
    out = coarse
    for d, t in zip((2, 1, 0), tile):
        cell = torch.remainder(torch.arange(g.nmesh, device="cuda") + (t - 1) * g.nsub - g.nbuff, g.N)
        f = (cell.to(torch.float64) + 0.5) / g.block + 0.5
        i = torch.floor(f)
        u = f - i
        w = (-u ** 3 / 2 + u * u - u / 2, 1.5 * u ** 3 - 2.5 * u * u + 1, -1.5 * u ** 3 + 2 * u * u + u / 2, u ** 3 / 2 - u * u / 2)
        shape = [1, 1, 1]
        shape[d] = g.nmesh
        out = sum(w[a].view(shape) * out.index_select(d, torch.remainder(i.long() + a - 2, g.M)) for a in range(4))
    return out


def _exact_split(case, seed):
    g = _geometry(case, seed)
    tile = tuple(1 + (seed // case["ntile"] ** q) % case["ntile"] for q in range(3))
    noise, cd, cp = _exact_coarse(g)
    n = g.nmesh
    cell = [torch.remainder(torch.arange(n, device="cuda") + (t - 1) * g.nsub - g.nbuff, g.N) for t in tile]
    res = torch.zeros((2 * n,) * 3, dtype=torch.float64, device="cuda")
    blk = [c // g.block for c in cell]
    for z in range(n):
        idx = cell[0][None, :] + g.N * (cell[1][:, None] + g.N * cell[2][z])
        mean = noise[blk[2][z]][blk[1]][:, blk[0]] / math.sqrt(float(g.block) ** 3)
        res[z, :n, :n] = _noise(idx.view(-1), g.seed).view(n, n) - mean
    box = 2 * n * g.alatt
    dk = 2 * math.pi / box
    k = _waves(2 * n, box, torch.float64)
    spec = torch.fft.rfftn(res)
    del res
    spec = _planes(spec, k, dk, lambda k2, x, y, z: _amplitude(k2, dk, 2 * n))
    safe = lambda k2: torch.where(k2 == 0, torch.ones_like(k2), k2)  # noqa: E731
    cut = lambda a: _irfftn(a, 2 * n)[:n, :n, :n].clone()  # noqa: E731
    eta = tuple(cut(_planes(spec, k, dk, lambda k2, x, y, z: 1j * (x, y, z)[q] / safe(k2))) + _interpolated(cp[q], g, tile)
                for q in range(3))
    delta = cut(spec) + _interpolated(cd, g, tile)
    del spec
    eta2, lap = _second(delta, n * g.alatt, case["ilpt"], case["lapd"], True)
    return dict(delta=delta, eta=eta, eta2=eta2, lapd=lap)


def exact(case, seed):
    """What run() returns, in 64 bits.  The shell analysis (alone or in a whole
    tile) and the merge walk shell by shell and halo by halo: in plain torch
    they take minutes, so they have no value here."""
    kind = case["kind"]
    if kind == "fields":
        return _exact_fields(case, int(seed))
    if kind == "split":
        return _exact_split(case, int(seed))
    if kind == "coarse":
        noise, delta, psi = _exact_coarse(_geometry(case, int(seed)))
        return dict(noise=noise, delta=delta, psi=psi)
    if kind == "peaks" and _inner(case) * (case["alatt"] / case["rf_min"]) ** 3 < 1e5:
        # a few thousand peaks; among more, near-ties of neighbouring cells
        # make the list of 64-bit fields another one
        fcrit = TileDriver(_config(case)).filter_fcrit()
        p = _find(_delta(case, int(seed)).to(torch.float64), case, fcrit, case["lapd"])
        return dict(delta_s=_rows(p.delta_s, _capacity(case)), lapd_s=_rows(p.lapd_s, _capacity(case)))
    return None
