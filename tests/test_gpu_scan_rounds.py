"""hs_scan_u32 at the edges of its tiles and rounds: every tile size, inputs that end
in a tile, on its edge and one element past it, one workgroup, misaligned scratch,
in place, every barrier kind."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILE = 4096


@pytest.mark.parametrize("round_bytes", [64 << 20, 16 << 20, 4 << 20])
@pytest.mark.parametrize("n", [1, 255, TILE, TILE + 1, 256 * TILE - 1, 256 * TILE + 1, 3 * 256 * TILE + 7, (3 << 22) + 1,
                               40_000_003])
def test_scan_rounds(hs, arena, n, round_bytes):
    import torch
    x = torch.empty(n + 4, dtype=torch.int32, device="cuda")[:n]
    hs.gen_uniform_u32(x, n, 0, 2**32 - 1)
    host = x.cpu().numpy().view(np.uint32)
    want = np.cumsum(host, dtype=np.uint64).astype(np.uint32)
    scratch = torch.empty(2 * 768 + 1, dtype=torch.int32, device="cuda")
    old = hs.get_scan_round_bytes()
    hs.set_scan_round_bytes(round_bytes)
    try:
        for wgs, off in ((0, 0), (0, 1), (1, 1), (2, 1), (3, 0), (30, 1), (512, 1), (768, 0)):
            for inclusive in (True, False):
                out = torch.full((n + 8,), -9, dtype=torch.int32, device="cuda")
                hs.scan_u32(arena, x, inclusive=inclusive, out=out[:n], num_wgs=wgs, scratch=scratch[off:])
                got = out.cpu().numpy().view(np.uint32)
                assert np.array_equal(got[:n], want if inclusive else want - host), (wgs, off, inclusive)
                assert (out[n:] == -9).all()
        for kind in ("flat", "two_level", "lf", "tree", "coop", "naive_all"):
            assert np.array_equal(hs.scan_u32(arena, x, barrier=kind).cpu().numpy().view(np.uint32), want), kind
        hs.scan_u32(arena, x, out=x)
        assert np.array_equal(x.cpu().numpy().view(np.uint32), want)
    finally:
        hs.set_scan_round_bytes(old)
