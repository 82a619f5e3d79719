"""hs_scan_u32 with a grid of the caller's: the grids that are served and refused,
and the scans of grids on both sides of one workgroup per CU."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_scan_grids(hs, arena):
    import torch
    cus = hs.device_info()["num_cus"]
    n = 3 * 32768 * 20 + 5  # several rounds of the small grids
    x = torch.empty(n, dtype=torch.int32, device="cuda")
    hs.gen_uniform_u32(x, 31, 0, 2**32 - 1)
    want = np.cumsum(x.cpu().numpy().view(np.uint32), dtype=np.uint32)
    for kind, most in (("xcd", 3), ("flat", 4), ("two_level", 4), ("coop", 4)):
        for wgs in (1, 2, 7, 20, 61, cus - 1, cus, cus + 1, most * cus):
            out = hs.scan_u32(arena, x, barrier=kind, num_wgs=wgs)
            assert np.array_equal(out.cpu().numpy().view(np.uint32), want), (kind, wgs)
        with pytest.raises(hs.HSError) as e:
            hs.scan_u32(arena, x, barrier=kind, num_wgs=most * cus + 1)
        assert e.value.status == 3, kind
