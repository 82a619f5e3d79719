"""Batches whose segments share tiles, cut them, or miss them: the heads of a
tile, its edges, empty segments and the line between the small and large tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SMALL, LARGE, FROM = 16384, 65536, 3 << 22  # scan tiles and where the large ones begin


def _off(lens, start=0):
    return (np.concatenate([[0], np.cumsum(np.asarray(lens, np.int64))]) + start).astype(np.uint64)


def _random(seed, nseg, top):
    rng = np.random.default_rng(seed)
    lens = np.exp2(rng.uniform(0, top, nseg)).astype(np.int64)
    lens[::5] = 0
    return lens


CASES = {
    "ones": _off(np.ones(70000 // 2, np.int64)),
    "one_element": _off([1], 3),
    "empty_ends": _off([0, 0, 5, 0, SMALL - 5, 0, 0]),
    "heads_at_tile_edges": _off([SMALL, SMALL - 1, 1, 1, SMALL - 1, 2 * SMALL + 1], 0),
    "start_off_by_one": _off([7, 250, 1, 2, 253, SMALL, 3], 1),
    "start_off_by_three": _off([1, 0, 255, 256, 257, 3 * SMALL], SMALL + 3),
    "short_rows": _off(_random(1, 65536, 6), 2),
    "ragged": _off(_random(2, 900, 17), 1),
    "below_large": _off([FROM - 4]),
    "at_large": _off([1, FROM - 1]),
    "large_with_heads": _off(np.concatenate([[LARGE - 1, 1, LARGE, 5], _random(3, 3000, 13), [FROM]]), 3),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_flat_batch_vs_oracle(hs, name):
    import torch
    off = CASES[name]
    a, n = int(off[0]), int(off[-1])
    x = torch.empty(n + 9, dtype=torch.int32, device="cuda")
    hs.gen_uniform_u32(x, 17, 0, 2**32 - 1)
    host = x.cpu().numpy().view(np.uint32)
    flat = np.concatenate([np.zeros(1, np.uint64), np.cumsum(host[:n], dtype=np.uint64)])  # sums of the first i
    at = off.astype(np.int64)
    sums = hs.reduce_batch_i32(x, off).cpu().numpy().view(np.uint32)
    assert np.array_equal(sums, (flat[at[1:]] - flat[at[:-1]]).astype(np.uint32))
    base = np.repeat(flat[at[:-1]], np.diff(at))
    for inclusive in (True, False):
        out = torch.full_like(x, -7)
        hs.scan_batch_u32(x, off, inclusive=inclusive, out=out)
        got = out.cpu().numpy().view(np.uint32)
        want = (flat[a + 1:n + 1] if inclusive else flat[a:n]) - base
        assert np.array_equal(got[a:n], want.astype(np.uint32)), inclusive
        assert (out[:a] == -7).all() and (out[n:] == -7).all()  # nothing outside the batch is written
    hs.scan_batch_u32(x, off, out=x)  # in place
    assert np.array_equal(x.cpu().numpy().view(np.uint32)[a:n], (flat[a + 1:n + 1] - base).astype(np.uint32))
