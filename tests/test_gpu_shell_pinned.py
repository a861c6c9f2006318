"""Launch parameters that were set hold whatever the batch: with one lane per
peak (post_width 1) and no wave post (coop_m above every m), a few peaks (too
few for a walk table), some thousand and some ten thousand go through the same
Float64 arithmetic, so the post's outputs have the same bits.  (Sbar, Sbar2 and
d2F are summed by the finish pass, whose waves per peak follow the batch.)"""
import numpy as np
import pytest

from peakpatch_hip import SHELL_PERSISTENT, collapse
from test_gpu_shell import FIELDS, bump_field

pytestmark = pytest.mark.gpu

POST = tuple(q for q in FIELDS if q not in ("Sbar", "Sbar2", "d2F"))


def test_pinned_post(ctx):
    n, p = 64, 50
    d, eta, eta2, lap = bump_field(n, 5)
    ct = collapse.sinusoidal_table()
    ctx.upload_collapse_table(ct.table, *ct.bounds)
    ctx.build_shell_tables(14)
    rng = np.random.default_rng(2)
    c = np.argsort(d[6:-6, 6:-6, 6:-6].ravel())[-4 * p::4]
    k, j, i = (q + 6 for q in np.unravel_index(c, (n - 12,) * 3))
    Rf = rng.uniform(4.0, 6.0, p)
    pk = dict(i=i.astype(np.int32), j=j.astype(np.int32), k=k.astype(np.int32), Rf=Rf,
              ir2min=np.floor((1.75 * Rf) ** 2).astype(np.int64), ZZon=rng.uniform(0.3, 0.8, p))

    def run(times):
        q = {a: np.tile(v, times) for a, v in pk.items()}
        return ctx.analyse_peaks(d, eta, q["i"], q["j"], q["k"], q["Rf"], q["ir2min"], q["ZZon"], 0.7, 1.0,
                                 eta2=eta2, lapd=lap, nbuff=2, kernel=SHELL_PERSISTENT)

    before = ctx.tunables()
    try:
        ctx.tunables(post_width=1, coop_m=1 << 20)
        want = run(1)
        ok = want["status"] == 0
        assert ok.sum() > 10 and (want["nshells"] > 64).sum() > 10
        for times in (40, 800):
            got = run(times)
            for f in POST:
                a = got[f].reshape(times, *want[f].shape)[:, ok]
                np.testing.assert_array_equal(a, np.broadcast_to(want[f][ok], a.shape), err_msg=f"{f} {times}")
    finally:
        ctx.tunables(**before)
    assert ctx.tunables() == before
