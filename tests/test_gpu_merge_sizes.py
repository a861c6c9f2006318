"""pp_merge_halos where its grid of cells and its rounds can go wrong: one
halo, a few, all in one place, on a line and in a plane, one far away, one
larger than the catalogue, long chains of exclusion, radii of zero and below.
The surviving set is the oracle's; the radius agrees to one Float32 ulp (the
caps are summed in another order, 1e-13 of the volume at most here, and a
radius is rounded to Float32 once)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from peakpatch_hip.api import Context
    return Context(0)


def _shape(name, n, rng):
    p = rng.uniform(-40.0, 40.0, (n, 3))
    r = 1.2 * (1.0 - rng.random(n)) ** (-1 / 3.2)
    if name == "point":
        p[:] = p[0]
    elif name == "line":
        p[:, 1:] = p[0, 1:]
        p[:, 0] *= 10
    elif name == "plane":
        p[:, 2] = p[0, 2]
    elif name == "far":
        p[n // 2] = (4e5, -3e5, 1e5)
    elif name == "giant":
        r[n // 3] = 60.0
    elif name == "chain":  # each halo inside the one before it only
        p[:] = 0.0
        p[:, 1] = np.arange(n)
        r = 1.5 - np.arange(n) * (0.4 / n)
    elif name == "signs":
        r[::3] = 0.0
        r[1::7] = -1.0
    elif name == "lattice":  # halos on the faces of cells, equal radii
        m = int(np.ceil(n ** (1 / 3)))
        p = np.stack(np.unravel_index(np.arange(n), (m, m, m)), 1) * 2.0
        r[:] = 1.5
    return p, r


@pytest.mark.parametrize("name", ["box", "point", "line", "plane", "far", "giant", "chain", "signs", "lattice"])
@pytest.mark.parametrize("n", [1, 2, 65, 700])
def test_merge_shapes(ctx, monkeypatch, name, n):
    from oracle import merger as OM
    from peakpatch_hip import catalog
    p, r = _shape(name, n, np.random.default_rng(n))
    rec = np.zeros((n, 11), np.float32)
    rec[:, :3], rec[:, 6] = p, r
    rec[:, 7] = np.arange(n)
    if name == "signs" and n == 1:
        with pytest.raises(Exception, match="degenerate catalogue extent"):
            catalog.merge_catalog(ctx, rec)
        return
    # every halo a candidate: the oracle's walk over 256^3 cells takes minutes here
    monkeypatch.setattr(OM.SpatialHash, "around", lambda self, c, dcell: range(1, len(self.ll)))
    alive, nr = OM.merge(rec[:, 0], rec[:, 1], rec[:, 2], rec[:, 6])
    want = rec[alive].copy()
    want[:, 6] = nr[alive].astype(np.float32)
    got = catalog.merge_catalog(ctx, rec)
    np.testing.assert_array_equal(got[:, 7], want[:, 7])
    assert np.all(np.abs(got[:, 6] - want[:, 6]) <= np.spacing(want[:, 6]))
