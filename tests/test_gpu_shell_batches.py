"""The shell analysis of the same peaks in batches of different sizes.  The
number of waves that gather and finish a peak (8, 4, 2, 1), the lanes that
post-process it (16 .. 1) and the walk table's widths follow the batch size,
so a peak repeated until each rule changes must keep its result.

The gather's bins see the same Float32 sums in the same order whatever the
waves: nshells, status and every decision are equal.  Float64 sums over at
most a few hundred shells or cells are grouped by lanes: 500 x 1.1e-16 of the
sum of magnitudes, 1e-11 of a column's largest value with room for the
division by a difference in the interpolation to R_TH.
"""
import numpy as np
import pytest

from peakpatch_hip import SHELL_PERSISTENT, collapse
from test_gpu_shell import FIELDS, bump_field

pytestmark = pytest.mark.gpu


def _run(ctx, fields, pk, times, lapd):
    d, eta, eta2, lap = fields
    rep = {k: np.tile(v, times) for k, v in pk.items()}
    mask = np.zeros(d.shape, np.int8)
    r = ctx.analyse_peaks(d, eta, rep["i"], rep["j"], rep["k"], rep["Rf"], rep["ir2min"], rep["ZZon"], 0.7, 1.0,
                          eta2=eta2 if lapd else None, lapd=lap if lapd else None, nbuff=2, mask=mask,
                          kernel=SHELL_PERSISTENT)
    return r, mask


@pytest.mark.parametrize("lapd", [False, True])
def test_batch_sizes(ctx, lapd):
    n = 64
    fields = bump_field(n, 5)
    ct = collapse.sinusoidal_table()
    ctx.upload_collapse_table(ct.table, *ct.bounds)
    ctx.build_shell_tables(14)
    rng = np.random.default_rng(2)
    p = 400
    d = fields[0]
    c = np.argsort(d[6:-6, 6:-6, 6:-6].ravel())[-4 * p::4]  # high cells: most collapse
    k, j, i = (q + 6 for q in np.unravel_index(c, (n - 12,) * 3))
    Rf = rng.uniform(2.5, 6.0, p)
    pk = dict(i=i.astype(np.int32), j=j.astype(np.int32), k=k.astype(np.int32), Rf=Rf,
              ir2min=np.floor((1.75 * Rf) ** 2).astype(np.int64), ZZon=rng.uniform(0.3, 0.8, p))
    pk["i"][:8], pk["j"][:8] = 2, 3  # spheres that leave the grid
    want, mask = _run(ctx, fields, pk, 1, lapd)
    ok = want["status"] == 0
    assert 0.2 * p < ok.sum() < p and (want["nshells"] > 16).sum() > 0.9 * p
    for times in (30, 100, 600):  # 12 k, 40 k, 240 k peaks: 4, 2, 1 waves on 256 CUs
        got, m = _run(ctx, fields, pk, times, lapd)
        np.testing.assert_array_equal(m, mask)
        for f in ("status", "nshells"):
            np.testing.assert_array_equal(got[f].reshape(times, p), np.broadcast_to(want[f], (times, p)))
        for f in FIELDS:
            a, b = got[f].reshape(times, *want[f].shape)[:, ok], want[f][ok]
            assert np.all(np.abs(a - b) <= 1e-11 * np.abs(b).max()), (f, times, float(np.abs(a - b).max()))
