"""The largest inner cube pp_find_peaks_field_noalloc takes, 8387136 row words,
and one of four words more, which it refuses."""
import ctypes as C

import pytest

from peakpatch_hip import _lib as L

pytestmark = pytest.mark.gpu


def test_largest_and_next(ctx):
    import torch
    n3, n2, n1 = 14563, 578, 3
    d = torch.zeros((n3, n2, n1), device="cuda")
    m = torch.zeros((n3, n2, n1), dtype=torch.int8, device="cuda")
    at = [(3, 4, 1), (n3 - 2, n2 - 2, 1)]
    for q in at:
        d[q] = 2.0
    o = [torch.zeros(8, dtype=torch.int32, device="cuda") for _ in range(4)]
    v = torch.zeros(8, device="cuda")
    pk = L.Peaks(8, 0, 0, *(a.data_ptr() for a in o), v.data_ptr(), None)
    torch.cuda.synchronize()

    def call(n2, n3):
        return ctx.lib.pp_find_peaks_field_noalloc(ctx.h, d.data_ptr(), m.data_ptr(), n1, n2, n3, 1, C.c_float(1.0), 0,
                                                   C.byref(pk))

    assert call(n2, n3) == 0 and pk.count == 2
    assert [(int(o[2][q]), int(o[1][q]), int(o[0][q])) for q in range(2)] == at
    assert call(2742, 3063) == -1 and b"scratch" in ctx.lib.pp_last_error()  # refused before any access
