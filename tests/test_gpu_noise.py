"""The device's Gaussian normals (pp_fill_noise_threefry) and their sums over
coarse cells (pp_coarse_create) against the oracle's Float64 normals.

Both sides are right to 1e-15 of a normal's radius (at most 8.6), so a value
rounded to Float32 is the oracle's or its neighbour, the neighbour for one in
10^6 (1e-15 of a Float32 spacing of 6e-8, times the values near zero).  A
coarse cell's Float64 sum of at most 130^3 normals is right to 2e-10 of its
norm in any order: one Float32 spacing.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from peakpatch_hip.api import Context
    return Context(0)


def _normals(n3, seed):
    from oracle import fields as OF
    g = OF.threefry_gaussian(seed, np.arange((n3 + 1) // 2, dtype=np.uint64))
    return np.stack(g, 1).reshape(-1)[:n3]


@pytest.mark.parametrize("n,seed", [(1, 0), (100, 5), (101, 2 ** 63 + 11)])
def test_normals(ctx, n, seed):
    want = _normals(n ** 3, seed).astype(np.float32).reshape((n,) * 3)
    got = ctx.fill_noise(n, seed)
    ctx.synchronize()
    got = got.cpu().numpy()
    assert np.all(np.abs(got - want) <= np.spacing(np.abs(want)))
    assert (got != want).sum() <= 2 + 4e-6 * want.size


@pytest.mark.parametrize("M,block", [(16, 1), (8, 2), (4, 3), (3, 16), (2, 41), (2, 130)])
def test_coarse_noise(ctx, M, block):
    from peakpatch_hip import split
    N = M * block
    cf = split.CoarseField(ctx, split.SplitGeom(N, 0, 1, M, 1.0, seed=9))
    noise = cf.download()[0]
    cf.close()
    want = _normals(N ** 3, 9).reshape(M, block, M, block, M, block).sum((1, 3, 5)) / np.sqrt(float(block) ** 3)
    want = want.astype(np.float32)
    assert noise.shape == want.shape
    assert np.all(np.abs(noise - want) <= np.spacing(np.abs(want)))
