"""The admission footprint of a served tile against the device memory a slot
takes: free memory before the slot's first tile less the least seen while it
runs two.  Meshes on line transforms and on rocFFT."""
import threading
import time

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("n", [192, 310, 320])
def test_a_slot_stays_within_its_footprint(homeltab_path, split, n):
    import torch
    from peakpatch_hip import collapse, serve
    r = serve.GpuTileRunner(table=collapse.read_homeltab(homeltab_path), split=split, trim_n=0)
    st = r.make_slot()
    if split:
        r.coarse(st["ctx"], n)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    seen, stop = [free], threading.Event()

    def watch():
        while not stop.is_set():
            seen.append(torch.cuda.mem_get_info()[0])
            time.sleep(0.0005)

    t = threading.Thread(target=watch)
    t.start()
    try:
        for q in range(2):
            out = r.run(st, serve.TileRequest(q, n, (0.0, 0.0, 0.0), seed=5 + q, tile=(1, 2, 1)))
        torch.cuda.synchronize()
        seen.append(torch.cuda.mem_get_info()[0])
    finally:
        stop.set()
        t.join()
        r.release_slot(st)
        r.close()
        torch.cuda.empty_cache()
    assert out.npeaks > 1000
    assert free - min(seen) <= r.footprint(n), ((free - min(seen)) / n ** 3, r.footprint(n) / n ** 3)
