"""The k^2 field (wsmooth = 3) of spectra whose power lies where the window is
far below its largest value: no mode may be left out."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,R", [(32, 8.0), (45, 9.0), (34, 8.0)])  # lines, odd lines, rocFFT
def test_far_modes_count(ctx, n, R):
    """A spectrum that starts where the window has fallen below 1e-15."""
    box = float(n)
    x = np.arange(n) * 2 * math.pi / n
    i = n // 2 - 3
    k = 2 * math.pi * i / box
    w = math.exp(-(k * R / 2) ** 2 / 2) * k * k
    assert 1e-35 < w < 1e-15
    spec = np.zeros((n, n, n // 2 + 1), np.complex64)
    spec[0, 0, i] = 1e15
    want = 2 * 1e15 * w * np.cos(i * x) / n ** 3
    got = ctx.smooth_field(spec, n, box, R, 3)
    assert np.abs(got - want[None, None, :]).max() <= 2e-5 * np.abs(want).max()


def test_peaks_of_a_field_of_far_modes(ctx):
    """pp_find_peaks on a plane wave: its k^2 field at the peaks is what the
    forward transform left of the wave and of its rounding, the same modes as
    pp_smooth_field's."""
    n, box = 32, 32.0
    x = np.arange(n) * 2 * math.pi / n
    d = np.ascontiguousarray(np.broadcast_to(np.cos(8 * x), (n, n, n)).astype(np.float32))
    R = [6.5, 2.0]
    pk = ctx.find_peaks(d, box, R, [-1.0, 0.01], want_lapd=True, nbuff=2)
    assert len(pk) > 100
    spec = ctx.rfft(d)
    for f in range(2):
        q = np.asarray(pk.filt) == f
        s = ctx.smooth_field(spec, n, box, R[f], 3)
        np.testing.assert_array_equal(pk.lapd_s[q], s[pk.k[q], pk.j[q], pk.i[q]])
