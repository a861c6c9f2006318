"""Halos with a NaN coordinate or radius in pp_merge_halos: kept as they are,
the rest merged as if they were not there (the reference's comparisons with
them are all false)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("on_device", [False, True])
@pytest.mark.parametrize("column", [0, 1, 2, 6])
def test_nan_halos(ctx, column, on_device):
    import torch
    from peakpatch_hip import catalog
    rng = np.random.default_rng(column)
    n = 3000
    rec = np.zeros((n, 11), np.float32)
    rec[:, :3] = rng.uniform(-20.0, 20.0, (n, 3))
    rec[:, 6] = np.minimum(1.2 * (1.0 - rng.random(n)) ** (-1 / 3.2), 6.0)
    rec[:, 7] = np.arange(n)
    bad = rng.random(n) < 0.02
    bad[:2] = True
    rec[1, :3], rec[1, 6] = rec[2, :3], 30.0  # would exclude most of the rest
    rec[bad, column] = np.nan
    merge = lambda r: (catalog.merge_catalog(ctx, torch.as_tensor(r, device="cuda")).cpu().numpy() if on_device
                       else np.asarray(catalog.merge_catalog(ctx, r)))
    got, want = merge(rec), merge(rec[~bad])
    is_bad = bad[got[:, 7].astype(int)]
    assert is_bad.sum() == bad.sum() and 100 < len(want) < 2900
    if column == 6:
        assert np.isnan(got[is_bad, 6]).all()
    else:
        r = rec[bad, 6]
        assert np.all(np.abs(got[is_bad, 6] - r) <= np.spacing(r))
    rest = got[~is_bad]
    np.testing.assert_array_equal(rest[:, 7], want[:, 7])
    assert np.all(np.abs(rest[:, 6] - want[:, 6]) <= np.spacing(want[:, 6]))
