"""The filter bank's spectra in padded rows (powers of two from 256 on) against
pp_smooth_field, whose rows are plain: the same rocFFT kernels at other
strides, so the filtered field at the peaks has the same bits.  Beside them
sizes that keep plain rows, and one size after the other on one context."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from peakpatch_hip.api import Context
    return Context(0)


@pytest.mark.parametrize("n,wsmooth", [(128, 1), (256, 1), (256, 0), (250, 1), (512, 1)])
def test_peaks_field(ctx, n, wsmooth):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    d = torch.randn((n, n, n), generator=g, device="cuda")
    box, R, fc = float(n), [4.0, 2.0], [0.01, 0.05]
    pk = ctx.find_peaks(d, box, R, fc, wsmooth=wsmooth, nbuff=2, max_peaks_per_filter=200000)
    assert len(pk) > 100
    dk = ctx.rfft(d.cpu().numpy())
    for f in range(2):
        s = ctx.smooth_field(dk, n, box, R[f], wsmooth)
        q = np.asarray(pk.filt) == f
        assert q.any()
        np.testing.assert_array_equal(pk.delta_s[q], s[pk.k[q], pk.j[q], pk.i[q]])
