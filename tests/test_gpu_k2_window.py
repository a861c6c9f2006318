"""The k^2-Gaussian window (wsmooth = 3) mode by mode: pp_smooth_field of a
spectrum of one mode, exact at the origin.

With ky = 0, n / 4 or n / 2 the rows y = 0 and 1 join without a rounding, every
twiddle at the origin is 1 and 1 / n^3 is a power of two, so the field there is
twice the window's Float32 value over n^3.  That value is the Float64 window
rounded once: at most half a spacing from it, 0.51 with the Float64 rounding
of the exponent."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16, 64])  # every radix-2 form: stages in LDS, stages in registers
def test_window_of_single_modes(ctx, n):
    box, worst = 1.3 * n, 0.0
    rng = np.random.default_rng(n)
    dk = 2.0 * math.pi / box
    for R in (0.7, 3.1, 0.11 * box):
        for _ in range(12):
            kx, ky, kz = int(rng.integers(1, n // 2)), int(rng.choice([0, n // 4, n // 2])), int(rng.integers(0, n))
            fy, fz = ky if ky < n // 2 else ky - n, kz if kz < n // 2 else kz - n
            k = math.sqrt((kx * dk) ** 2 + (fy * dk) ** 2 + (fz * dk) ** 2)
            want = math.exp(-(k * R / 2) ** 2 / 2) * k * k
            if not want > 1e-30:  # Float32's small end: fewer digits
                continue
            spec = np.zeros((n, n, n // 2 + 1), np.complex64)
            spec[kz, ky, kx] = 1.0
            got = float(ctx.smooth_field(spec, n, box, R, 3)[0, 0, 0]) * n ** 3 / 2
            err = abs(got - want) / float(np.spacing(np.float32(want)))
            worst = max(worst, err)
            assert err <= 0.51, (R, kx, fy, fz, got, want, err)
    assert worst > 0
