"""The scan's tiles at the line between the small and the large ones, with heads on the
edges of the large ones, ends that cut them, and more tiles than workgroups."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LARGE, FROM = 32768, 7 << 22


@pytest.mark.parametrize("start", [0, 1])
@pytest.mark.parametrize("total", [FROM - 1, FROM, FROM + 1, 2 * FROM + 12345])
def test_line_between_the_tiles(hs, start, total):
    import torch
    lens = [LARGE, LARGE - 1, 1, 0, 2 * LARGE + 1, 5, 1, 1, 255, 256, 257, 3 * LARGE]
    off = np.concatenate([[0], np.cumsum(lens + [total - sum(lens)])]).astype(np.uint64) + np.uint64(start)
    n = int(off[-1])
    x = torch.empty(n + 5, dtype=torch.int32, device="cuda")
    hs.gen_uniform_u32(x, 41, 0, 2**32 - 1)
    host = x.cpu().numpy().view(np.uint32)
    for inclusive in (True, False):
        out = torch.full_like(x, -7)
        hs.scan_batch_u32(x, off, inclusive=inclusive, out=out)
        got = out.cpu().numpy().view(np.uint32)
        for a, b in zip(off[:-1].astype(int), off[1:].astype(int)):
            want = np.cumsum(host[a:b], dtype=np.uint32)
            assert np.array_equal(got[a:b], want if inclusive else want - host[a:b]), (a, b, inclusive)
        assert (out[:start] == -7).all() and (out[n:] == -7).all()
