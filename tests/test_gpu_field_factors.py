"""The transfer factors of the field kernels: wave numbers, 1 / k^2, the
amplitude and the constants of the fields, whatever the units.

With P = A / k^3 the density does not depend on the unit of length and the
displacements scale with it, so two units whose wave numbers round to Float32
in opposite directions show what the factors lose: the transforms round alike
in both.  A mode's product with its factor is rounded once (2^-24 at most,
2.1e-8 rms, another way in every mode), and a hundred modes or more carry a
field, so the fields' sizes may differ by 3 x sqrt(2) x 2.1e-8 / 10 = 9e-9 of
the ratio of the units; a constant rounded to Float32 makes up to 6e-8 each.
"""
import ctypes as C
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GAIN = 9e-9


def _power(k):
    return 0.01 * k ** -3.0


def _round_off(v):
    return float(np.float32(v)) / v - 1.0


def _units(n, cell):
    """Two lengths of a cell, near to 1 and to 1.5 times `cell`, at which
    2 pi / (n cell) and its inverse square over n^3 round up and down by the
    most."""
    out = []
    for c, sign in ((cell, 1.0), (1.5 * cell, -1.0)):
        b = n * c * np.linspace(0.9, 1.1, 4001)
        score = [sign * (_round_off(2 * math.pi / v) + _round_off((v / (2 * math.pi)) ** 2 / float(n) ** 3)) for v in b]
        out.append(float(b[int(np.argmax(score))]) / n)
    return out


def _gain(got, want, ratio):
    g, w = (a.cpu().numpy().astype(np.float64) for a in (got, want))
    return float((g * w).sum() / (w * w).sum() / ratio - 1.0)


@pytest.mark.parametrize("n", [60, 63, 64])
def test_periodic_factors(ctx, n):
    from peakpatch_hip import synth
    c = _units(n, 1.3)
    a, b = (synth.make_tile(ctx, n, n * u, seed=n, ilpt=2, want_lapd=False, pk=_power) for u in c)
    assert abs(_gain(b.delta, a.delta, 1.0)) <= GAIN
    for q in range(3):
        for name in ("eta", "eta2"):
            got = _gain(getattr(b, name)[q], getattr(a, name)[q], c[1] / c[0])
            assert abs(got) <= GAIN, (name, q, got)


@pytest.mark.parametrize("n", [48, 64, 60])
def test_split_factors(ctx, n):
    from peakpatch_hip import split
    c = _units(n, 1.3)  # the padded box's wave numbers are half the tile's

    def tile(u):
        cf = split.CoarseField(ctx, split.SplitGeom(n, 4, 2, 4, u, seed=n), pk=_power)
        t = split.make_split_tile(ctx, cf, 1, 2, 1, ilpt=2, want_lapd=True)
        cf.close()
        return t

    a, b = (tile(u) for u in c)
    r = c[1] / c[0]
    # (the displacements' power lies in the few modes of the coarse field)
    for name, x, y, s in [("delta", a.delta, b.delta, 1.0), ("lapd", a.lapd, b.lapd, r ** -2)]:
        got = _gain(y, x, s)
        assert abs(got) <= GAIN, (name, got)


@pytest.mark.parametrize("unit", [3.0857e22, 1e-12])  # metres to the Mpc; very small numbers
def test_units(ctx, unit):
    """Lengths in other units: the density stays, displacements scale."""
    import torch
    from peakpatch_hip import _lib as L
    from peakpatch_hip import synth
    n, box = 32, 40.0
    k, P = synth.pk_table()

    def fields(u):
        f = [torch.empty((n, n, n), device="cuda") for _ in range(7)]
        ku, Pu = np.ascontiguousarray(k / u), np.ascontiguousarray(P * u ** 3)
        tab = L.PkTable(len(ku), ku.ctypes.data, Pu.ctypes.data)
        out = L.TileFields(*(a.data_ptr() for a in f), None)
        ctx._call(lambda: ctx.lib.pp_make_tile_fields(ctx.h, n, box * u, 5, C.byref(tab), C.byref(out)), True)
        return [a.cpu().numpy().astype(np.float64) for a in f]

    want, got = fields(1.0), fields(unit)
    for q, (a, b) in enumerate(zip(got, want)):
        s = 1.0 if q == 0 else unit
        assert np.isfinite(a).all(), q
        assert np.abs(a / s - b).max() <= 2e-5 * np.abs(b).max(), q


@pytest.mark.parametrize("unit", [3.0857e22, 1e-12])
def test_units_split(ctx, unit):
    """The same for a split tile, with P = A / k^3, which its table continues
    to any k."""
    from peakpatch_hip import split

    def fields(u):
        cf = split.CoarseField(ctx, split.SplitGeom(32, 3, 2, 29, 0.9 * u, seed=3), pk=_power)
        t = split.make_split_tile(ctx, cf, 2, 1, 2, ilpt=2, want_lapd=False)
        cf.close()
        return [a.cpu().numpy().astype(np.float64) for a in (t.delta, *t.eta, *t.eta2)]

    want, got = fields(1.0), fields(unit)
    for q, (a, b) in enumerate(zip(got, want)):
        s = 1.0 if q == 0 else unit
        assert np.isfinite(a).all(), q
        assert np.abs(a / s - b).max() <= 2e-5 * np.abs(b).max(), q
