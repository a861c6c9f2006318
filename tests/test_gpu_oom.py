"""After a call that did not fit into device memory."""
import numpy as np
import pytest

from peakpatch_hip import Context, PPError

pytestmark = pytest.mark.gpu


def test_a_refused_call_leaves_no_error_behind():
    """A mesh that does not fit is refused as out of memory; the next call on
    the same context is not."""
    import torch
    d = np.random.default_rng(1).normal(size=(32, 32, 32)).astype(np.float32)
    with Context(0) as ctx:
        want = ctx.rfft(d)
        ctx.fill_noise(8, 1)
        ctx.synchronize()
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        held = torch.empty(torch.cuda.mem_get_info()[0] - (400 << 20), dtype=torch.uint8, device="cuda")
        try:
            big = np.broadcast_to(np.float32(0), (512, 512, 512))
            with pytest.raises(PPError, match="OOM"):
                ctx.find_peaks_field(np.ascontiguousarray(big), np.zeros(big.shape, np.int8), 2, 1.0)
            ctx.fill_noise(8, 1)
            np.testing.assert_array_equal(ctx.rfft(d), want)
        finally:
            del held
            torch.cuda.empty_cache()
