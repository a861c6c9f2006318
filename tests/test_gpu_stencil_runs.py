"""The peak stencil's tiles and runs of words (k_peak_bits, k_peak_emit) where
they can go wrong: inner cubes of one cell, one word and a bit more, one row,
one plane, planes that fill no tile, and so many words that a run is more than
256 of them; several calls on one context, whose state each call clears; the
cut at max_peaks inside and at the edge of a run.  Whole numbers throughout:
equal to the definition (PeakFind.jl:15-78) evaluated on shifted arrays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from peakpatch_hip.api import Context
    return Context(0)


def _field(shape, seed):
    # multiples of 1/8: plateaus, whose cells are all peaks
    return np.round(np.random.default_rng(seed).normal(size=shape) * 8).astype(np.float32) / 8


def _peaks(d, mask, nbuff, fcrit, max_peaks):
    n3, n2, n1 = d.shape
    ins = tuple(slice(nbuff, n - nbuff) for n in d.shape)
    top = np.full(d[ins].shape, -np.inf, np.float32)
    for a in (-1, 0, 1):
        for b in (-1, 0, 1):
            for c in (-1, 0, 1):
                top = np.maximum(top, d[nbuff + a:n3 - nbuff + a, nbuff + b:n2 - nbuff + b, nbuff + c:n1 - nbuff + c])
    k, j, i = np.nonzero((d[ins] >= fcrit) & (d[ins] >= top) & (mask[ins] != 1))
    k, j, i = (q[:max_peaks] + nbuff for q in (k, j, i))
    mask[k, j, i] = 1
    return i, j, k, d[k, j, i]


@pytest.mark.parametrize("shape,nbuff,fcrit,cut", [
    ((3, 3, 3), 1, -9.0, None), ((3, 3, 67), 1, -9.0, None), ((3, 40, 66), 1, -9.0, 5),
    ((37, 3, 131), 1, 0.5, None), ((8, 19, 200), 2, 0.5, 77), ((70, 33, 68), 1, -9.0, None),
    ((402, 402, 131), 1, 0.5, None), ((402, 402, 131), 1, 0.5, 300001)])
def test_stencil(ctx, shape, nbuff, fcrit, cut):
    d = _field(shape, sum(shape))
    mask = (np.random.default_rng(1).random(shape) < 0.2).astype(np.int8)
    want_mask, got_mask = mask.copy(), mask.copy()
    want = _peaks(d, want_mask, nbuff, fcrit, cut if cut else d.size)
    for _ in range(2):  # the second call finds none of the first one's peaks
        got = ctx.find_peaks_field(d, got_mask, nbuff, fcrit, max_peaks=cut if cut else d.size)
        assert len(got) == len(want[0])
        for a, b in zip((got.i, got.j, got.k, got.delta_s), want):
            np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(got_mask, want_mask)
        want = _peaks(d, want_mask, nbuff, fcrit, cut if cut else d.size)
