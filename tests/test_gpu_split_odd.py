"""Split tiles of odd nmesh: the residual's pairs of cells end one cell past the
tile, which has to stay zero.  Lengths with a line transform's factors and
without, against the oracle's isolated convolution, within 2e-5 of each
field's largest value (Float32 transforms against pocketfft in Float64, the
tolerance of the even sizes)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nmesh,nbuff,ntile,M,tile", [
    (13, 1, 2, 8, (2, 1, 2)), (25, 3, 2, 11, (1, 2, 1)), (27, 4, 3, 13, (3, 1, 2)), (33, 2, 2, 31, (2, 2, 2)),
    (63, 5, 2, 29, (1, 1, 2))])
def test_odd_split_tile(ctx, nmesh, nbuff, ntile, M, tile):
    from oracle import fields as OF
    from peakpatch_hip import split, synth
    g = split.SplitGeom(nmesh, nbuff, ntile, M, 1.1, seed=nmesh)
    cf = split.CoarseField(ctx, g)
    t = split.make_split_tile(ctx, cf, *tile, ilpt=2, want_lapd=True)
    ref = OF.split_tile(OF.SplitGeom(nmesh, nbuff, ntile, M, 1.1), *tile, nmesh, OF.PkTable(*synth.pk_table()))
    for name, got, want in [("delta", t.delta, ref.delta), ("lapd", t.lapd, ref.lapd),
                            *((f"eta{q}", t.eta[q], ref.eta[q]) for q in range(3)),
                            *((f"eta2{q}", t.eta2[q], ref.eta2[q]) for q in range(3))]:
        scale = float(np.abs(want).max())
        err = float(np.abs(got.cpu().numpy() - want).max())
        assert scale > 0 and err <= 2e-5 * scale, (name, err, scale)
    cf.close()
