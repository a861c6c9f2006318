"""Rounding of the k^2 field's transform (pp_smooth_field, wsmooth = 3) beside
the general one's: the same field from the spectrum times k^2 and the Gaussian
window (wsmooth = 0), which rocFFT transforms.  Both products and both
transforms are Float32, so the first may be no further from 64 bits than the
second; the rms over n^3 >= 4096 cells is certain to some 2 per cent, 5 are
allowed.  Every radix, even and odd lengths, stages in LDS and in registers."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16, 25, 27, 30, 45, 48, 60, 63, 64, 75, 81, 96, 98, 105, 120, 125, 128])
def test_no_further_off_than_the_general_transform(ctx, n):
    box, R = 1.0 * n, 1.7
    rng = np.random.default_rng(n)
    spec = np.fft.rfftn(rng.normal(size=(n, n, n))).astype(np.complex64)
    f = np.fft.fftfreq(n, 1.0 / n) * (2 * math.pi / box)
    k2 = (np.arange(n // 2 + 1) * (2 * math.pi / box)) ** 2 + f[:, None] ** 2 + f[:, None, None] ** 2
    gauss = np.exp(-k2 * R * R / 8)
    k2[0, 0, 0] = 1.0
    times = (spec * k2).astype(np.complex64)

    def error(got, a):
        a = np.fft.ifft(np.fft.ifft(a, axis=0), axis=1)
        want = np.fft.irfft(a, n=n, axis=2)
        return float(np.sqrt(((got - want) ** 2).mean() / (want ** 2).mean()))

    lines = error(ctx.smooth_field(spec, n, box, R, 3), spec * (k2 * gauss))
    general = error(ctx.smooth_field(times, n, box, R, 0), times * gauss)
    assert lines <= 1.05 * general, (lines, general)
