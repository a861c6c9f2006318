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
        big = torch.zeros((640, 640, 640), device="cuda")
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        held = torch.empty(torch.cuda.mem_get_info()[0] - (400 << 20), dtype=torch.uint8, device="cuda")
        try:
            with pytest.raises(PPError, match="OOM"):  # three arrays of 1 GB
                ctx.find_peaks(big, 640.0, [2.0], [1.0], nbuff=2)
            ctx.fill_noise(8, 1)
            np.testing.assert_array_equal(ctx.rfft(d), want)
        finally:
            del held, big
            torch.cuda.empty_cache()
