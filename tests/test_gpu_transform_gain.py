"""The field kernels' transforms keep the amplitude: with a constant P(k) the
density is the white noise times a constant, forward and back through every
stage of the line transforms on all three axes.

Read off by regression on the noise, the factor may be off by what the radix-8
butterfly's Float32 root takes (1.7e-8 of a quarter of the sums, at most three
stages, there and back, three axes: 7.7e-8); the random rounding of n^3 cells
and the twiddles, whose tables are rounded without a mean, add 3e-9.  Twiddles
rounded to the nearest take 1.1 to 1.5e-7 at these lengths."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [48, 96, 128, 192, 240, 256])
def test_white_noise_keeps_its_size(ctx, n):
    from peakpatch_hip import synth
    box, P0 = 1.1 * n, 0.37
    t = synth.make_tile(ctx, n, box, seed=n, ilpt=1, want_lapd=False, pk=lambda k: P0 + 0.0 * k)
    noise = ctx.fill_noise(n, n)
    ctx.synchronize()
    w = noise.double().cpu().numpy()
    w = (w - w.mean()) * math.sqrt(P0 * (2 * math.pi / box) ** 3 * float(n) ** 3)
    g = t.delta.double().cpu().numpy()
    gain = float((g * w).sum() / (w * w).sum() - 1.0)
    assert abs(gain) <= 8e-8, gain
    assert np.abs(g - w).max() <= 2e-5 * np.abs(w).max()
