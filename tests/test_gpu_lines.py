"""The field kernels on line transforms (csrc/pp_fft.h) at the lengths where
their stages and tiles can go wrong: the shortest and an odd one, every radix
alone and mixed, butterflies that do not divide the threads, tiles with a
remainder of columns, odd numbers of rows; and lengths without a line
transform, which take rocFFT.

Tolerance: 2e-5 of each field's largest value, as for the fields on rocFFT
(Float32 transforms against pocketfft in Float64).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _close(name, got, want):
    scale = float(np.abs(want).max())
    err = float(np.abs(got - want).max())
    assert scale > 0 and err <= 2e-5 * scale, (name, err, scale)


@pytest.mark.parametrize("n", [14, 16, 21, 27, 34, 35, 49, 60, 64, 75, 96, 98, 125, 128, 144])
def test_periodic_fields(ctx, n):
    from oracle import fields as OF
    from peakpatch_hip import synth
    box = 1.3 * n
    t = synth.make_tile(ctx, n, box, seed=n, ilpt=2, want_lapd=True)
    ref = OF.make_tile(n, box, n, OF.PkTable(*synth.pk_table()))
    host = lambda a: a.cpu().numpy()
    _close("delta", host(t.delta), ref.delta)
    _close("lapd", host(t.lapd), ref.lapd)
    for q in range(3):
        _close(f"eta{q}", host(t.eta[q]), ref.eta[q])
        _close(f"eta2{q}", host(t.eta2[q]), ref.eta2[q])


def test_uneven_power_table(ctx):
    """A P(k) table whose rows are not evenly spaced in log k."""
    import ctypes as C

    import torch
    from oracle import fields as OF
    from peakpatch_hip import _lib as L
    from peakpatch_hip import synth
    n, box = 40, 60.0
    k, P = synth.pk_table()
    pick = np.unique(np.concatenate([np.arange(0, 1200, 7), np.arange(1200, 2001, 3)]))
    k, P = np.ascontiguousarray(k[pick]), np.ascontiguousarray(P[pick])
    f = [torch.empty((n, n, n), device="cuda") for _ in range(4)]
    tab = L.PkTable(len(k), k.ctypes.data, P.ctypes.data)
    out = L.TileFields(*(a.data_ptr() for a in f), None, None, None, None)
    ctx._call(lambda: ctx.lib.pp_make_tile_fields(ctx.h, n, box, 5, C.byref(tab), C.byref(out)), True)
    ref = OF.make_tile(n, box, 5, OF.PkTable(k, P), ilpt=1, want_lapd=False)
    _close("delta", f[0].cpu().numpy(), ref.delta)
    for q in range(3):
        _close(f"eta{q}", f[1 + q].cpu().numpy(), ref.eta[q])


@pytest.mark.parametrize("nmesh,nbuff,ntile,M,tile,second", [
    (16, 2, 2, 14, (1, 2, 1), True),     # shortest line, block 2
    (18, 3, 3, 14, (3, 1, 2), True),     # block 3, lines no multiple of the threads' eight
    (30, 5, 4, 10, (2, 4, 3), True),     # 2 3 5
    (50, 5, 3, 13, (1, 3, 2), False),    # first order only
    (56, 4, 2, 8, (1, 1, 1), True),      # radix 7; the wrap in all three axes
    (96, 8, 2, 11, (2, 2, 1), True),     # 8 4 3
    (26, 2, 2, 8, (1, 2, 2), True),      # no line transform (factor 13): rocFFT
])
def test_split_tile(ctx, nmesh, nbuff, ntile, M, tile, second):
    from oracle import fields as OF
    from peakpatch_hip import split, synth
    g = split.SplitGeom(nmesh, nbuff, ntile, M, 1.1, seed=nmesh)
    cf = split.CoarseField(ctx, g)
    t = split.make_split_tile(ctx, cf, *tile, ilpt=2 if second else 1, want_lapd=second)
    ref = OF.split_tile(OF.SplitGeom(nmesh, nbuff, ntile, M, 1.1), *tile, nmesh, OF.PkTable(*synth.pk_table()))
    host = lambda a: a.cpu().numpy()
    _close("delta", host(t.delta), ref.delta)
    for q in range(3):
        _close(f"eta{q}", host(t.eta[q]), ref.eta[q])
        if second:
            _close(f"eta2{q}", host(t.eta2[q]), ref.eta2[q])
    if second:
        _close("lapd", host(t.lapd), ref.lapd)
    cf.close()


@pytest.mark.parametrize("n,nbuff", [(25, 2), (48, 1), (63, 5), (64, 4), (100, 9), (128, 30), (34, 3)])
def test_k2_field_at_the_peaks(ctx, n, nbuff):
    """The wsmooth = 3 field at the peaks of a bank of radii from below a cell
    (every mode kept) to a quarter of the box (few modes kept) and zero: the
    bits of pp_smooth_field, and the FP64 field within 2e-5 of its largest
    value (the Float32 transforms' noise over fewer modes than above)."""
    import torch
    from oracle import oracle as O
    box = 1.0 * n
    rng = np.random.default_rng(n)
    delta = rng.normal(size=(n, n, n)).astype(np.float32)
    Rf = np.array([0.25 * n, 0.1 * n, 3.0, 0.4, 0.0])
    fcrit = np.array([-1e30, -1e30, -1e30, 0.5, 0.5], np.float32)
    pk = ctx.find_peaks(torch.as_tensor(delta, device="cuda"), box, Rf, fcrit, want_lapd=True, nbuff=nbuff)
    assert set(pk.filt.tolist()) >= {1, 2, 3}
    dk = ctx.rfft(delta)
    for f, R in enumerate(Rf):
        at = pk.filt == f
        s = ctx.smooth_field(dk, n, box, R, 3)
        np.testing.assert_array_equal(pk.lapd_s[at], s[pk.k[at], pk.j[at], pk.i[at]])
        _close(f"R={R}", s, O.smooth_field(dk, n, box, R, 3))
