"""The field kernels' line transforms at the lengths that are served and at
those whose kernels or workgroups differ: multiples of 64 (first and last
stage in registers) with factors 2, 3 (192, 512, 576, 768, 1024), 5 and 7
(320, 448, 640, 896, 960), columns of 16 and of 8, workgroups of part of a wave
(576, 960), more than 64 KB of LDS (1000, 1024), stages in LDS (1000).

Fields against torch's transforms in Float64 on the device, from the same
Float32 noise (pp_fill_noise_threefry) and P = A / k^3, within 2e-5 of each
field's largest value, as for the short lengths; 64 and 128 as split tiles
against the oracle."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

A = 0.01


def _power(k):
    return A * k ** -3.0


def _close(name, got, want):
    scale = float(want.abs().max())
    err = float((got.double() - want).abs().max())
    assert scale > 0 and err <= 2e-5 * scale, (name, err, scale)


def _waves(n, box):
    """k along x (half), y and z in units of the grid, broadcastable."""
    import torch
    f = torch.arange(n, device="cuda")
    f = torch.where(f < (n + 1) // 2, f, f - n).double() * (2 * math.pi / box)
    x = torch.arange(n // 2 + 1, device="cuda").double() * (2 * math.pi / box)
    return x[None, :], f[:, None], f


def _back(spec, n):
    """Normalised inverse of a half spectrum, which is overwritten."""
    import torch
    for q in range(spec.shape[2]):  # a plane of kx at a time: the work space stays small
        spec[:, :, q] = torch.fft.ifft2(spec[:, :, q])
    spec[:, :, 0].imag.zero_()
    if n % 2 == 0:
        spec[:, :, -1].imag.zero_()
    out = torch.empty((n, n, n), dtype=torch.float64, device="cuda")
    for q in range(n):
        out[q] = torch.fft.irfft(spec[q], n=n, dim=1)
    return out


def _times(spec, k, fn, nyq=False):
    """A copy of spec with every kz plane times fn(kx, ky, kz, k^2), k = 0 and,
    with nyq, the Nyquist planes zeroed."""
    import torch
    n = spec.shape[0]
    out = torch.empty_like(spec)
    for q in range(n):
        kz = k[2][q]
        k2 = k[0] ** 2 + k[1] ** 2 + kz ** 2
        if q == 0:
            k2[0, 0] = 1.0
        out[q] = spec[q] * fn(k[0], k[1], kz, k2)
    out[0, 0, 0] = 0
    if nyq:
        out[:, :, n // 2] = 0
        out[:, n // 2] = 0
        out[n // 2] = 0
    return out


def _forward(a):
    import torch
    n = a.shape[0]
    spec = torch.empty((n, n, n // 2 + 1), dtype=torch.complex128, device="cuda")
    for q in range(n):
        spec[q] = torch.fft.rfft(a[q].double(), dim=1)
    for q in range(n // 2 + 1):
        spec[:, :, q] = torch.fft.fft2(spec[:, :, q])
    return spec


def _second_order(spec, k, n, split_rules, delta=None):
    """Source of the second order from a density's spectrum."""
    pair = ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))
    phi = lambda a, b: _back(_times(spec, k, lambda x, y, z, k2: -(x, y, z)[a] * (x, y, z)[b] / k2, split_rules), n)
    if split_rules:
        src = delta.double() ** 2 / 2
        for a, b in pair:
            src -= phi(a, b) ** 2 * (0.5 if a == b else 1.0)
        return src
    p, q, r = (phi(a, a) for a in range(3))
    src = p * q + p * r + q * r
    del p, q, r
    for a, b in pair[3:]:
        src -= phi(a, b) ** 2
    return src


@pytest.mark.parametrize("n", [192, 320, 448, 512, 576, 640, 768, 896, 960, 1000, 1024])
def test_periodic_lengths(ctx, n):
    import torch
    from peakpatch_hip import synth
    box = 1.3 * n
    t = synth.make_tile(ctx, n, box, seed=n, ilpt=2, want_lapd=True, pk=_power)
    ctx.lib.pp_ctx_release_scratch(ctx.h)
    noise = ctx.fill_noise(n, n)
    ctx.synchronize()
    k, dk = _waves(n, box), 2 * math.pi / box
    spec = _forward(noise)
    del noise
    spec = _times(spec, k, lambda x, y, z, k2: torch.sqrt(A * k2 ** -1.5 * dk ** 3 * float(n) ** 3))
    _close("delta", t.delta, _back(spec.clone(), n))
    _close("lapd", t.lapd, _back(_times(spec, k, lambda x, y, z, k2: k2 / float(n) ** 3), n))
    for q in range(3):
        _close(f"eta{q}", t.eta[q], _back(_times(spec, k, lambda x, y, z, k2: 1j * (x, y, z)[q] / k2, True), n))
    src = _second_order(spec, k, n, False)
    spec = _forward(src)
    del src
    for q in range(3):
        _close(f"eta2{q}", t.eta2[q], _back(_times(spec, k, lambda x, y, z, k2: -1j * (x, y, z)[q] / k2, True), n))
    del spec, t
    torch.cuda.empty_cache()


@pytest.mark.parametrize("nmesh,nbuff,ntile,M,tile", [(64, 6, 2, 29, (2, 1, 1)), (128, 10, 2, 59, (1, 2, 1))])
def test_split_tile_against_the_oracle(ctx, nmesh, nbuff, ntile, M, tile):
    from oracle import fields as OF
    from peakpatch_hip import split, synth
    g = split.SplitGeom(nmesh, nbuff, ntile, M, 1.1, seed=nmesh)
    cf = split.CoarseField(ctx, g)
    t = split.make_split_tile(ctx, cf, *tile, ilpt=2, want_lapd=True)
    ref = OF.split_tile(OF.SplitGeom(nmesh, nbuff, ntile, M, 1.1), *tile, nmesh, OF.PkTable(*synth.pk_table()))
    cf.close()
    for name, got, want in [("delta", t.delta, ref.delta), ("lapd", t.lapd, ref.lapd),
                            *((f"eta{q}", t.eta[q], ref.eta[q]) for q in range(3)),
                            *((f"eta2{q}", t.eta2[q], ref.eta2[q]) for q in range(3))]:
        scale = float(np.abs(want).max())
        err = float(np.abs(got.cpu().numpy() - want).max())
        assert scale > 0 and err <= 2e-5 * scale, (name, err, scale)


def _interpolated(coarse, n, nbuff, block):
    """Catmull-Rom interpolation of a coarse field onto the tile of a run of one
    tile, whose grid is the global one moved by nbuff."""
    import torch
    M = coarse.shape[0]
    cell = torch.remainder(torch.arange(n, device="cuda") - nbuff, n)
    f = (cell.double() + 0.5) / block + 0.5
    i = torch.floor(f)
    u = f - i
    w = (-u ** 3 / 2 + u * u - u / 2, 1.5 * u ** 3 - 2.5 * u * u + 1, -1.5 * u ** 3 + 2 * u * u + u / 2, u ** 3 / 2 - u * u / 2)
    out = coarse
    for d in range(3):
        shape = [1, 1, 1]
        shape[d] = n
        out = sum(w[a].view(shape) * out.index_select(d, torch.remainder(i.long() + a - 2, M)) for a in range(4))
    return out


@pytest.mark.parametrize("n,M", [(192, 24), (320, 40), (448, 56), (512, 64), (576, 36), (768, 48)])
def test_split_lengths(ctx, n, M):
    """A run of one tile: its cells are the whole global grid's."""
    import torch
    from peakpatch_hip import split
    nbuff, alatt, seed = 5, 0.9, n + 1
    g = split.SplitGeom(n, nbuff, 1, M, alatt, seed=seed)
    cf = split.CoarseField(ctx, g, pk=_power)
    t = split.make_split_tile(ctx, cf, 1, 1, 1, ilpt=2, want_lapd=True)
    cn, cd, cp = cf.download()
    cf.close()
    block = n // M
    fine = torch.roll(ctx.fill_noise(n, seed), (nbuff, nbuff, nbuff), (0, 1, 2))
    ctx.synchronize()
    torch.cuda.synchronize()
    blk = torch.remainder(torch.arange(n, device="cuda") - nbuff, n) // block
    mean = torch.as_tensor(cn, device="cuda").double() / math.sqrt(float(block) ** 3)
    pad = torch.zeros((2 * n,) * 3, dtype=torch.float32, device="cuda")
    for z in range(n):
        pad[z, :n, :n] = (fine[z].double() - mean[blk[z]][blk][:, blk]).float()
    del fine
    box = 2 * n * alatt
    k, dk = _waves(2 * n, box), 2 * math.pi / box
    base = _forward(pad)
    del pad
    amp = lambda k2: torch.sqrt(A * k2 ** -1.5 * dk ** 3 * float(2 * n) ** 3)
    whole = lambda a: torch.as_tensor(a, device="cuda").double()
    cut = lambda s: _back(s, 2 * n)[:n, :n, :n].clone()
    fields = [("delta", t.delta, cd, lambda x, y, z, k2: amp(k2)),
              *((f"eta{q}", t.eta[q], cp[q], lambda x, y, z, k2, q=q: 1j * (x, y, z)[q] / k2 * amp(k2)) for q in range(3))]
    for name, got, coarse, fn in fields if n <= 576 else fields[:2]:
        want = cut(_times(base, k, fn))
        torch.cuda.empty_cache()
        want += _interpolated(whole(coarse), n, nbuff, block)
        _close(name, got, want)
        del want
    del base
    torch.cuda.empty_cache()
    # the tile-periodic fields from the tile's own density
    k = _waves(n, n * alatt)
    spec = _forward(t.delta)
    _close("lapd", t.lapd, _back(_times(spec, k, lambda x, y, z, k2: k2, True), n))
    src = _second_order(spec, k, n, True, t.delta)
    spec = _forward(src)
    del src
    for q in range(3):
        _close(f"eta2{q}", t.eta2[q], _back(_times(spec, k, lambda x, y, z, k2: -1j * (x, y, z)[q] / k2, True), n))
    del spec, t
    torch.cuda.empty_cache()
