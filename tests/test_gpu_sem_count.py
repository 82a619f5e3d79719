"""Semaphores whose count is one atomic word: every unit comes back."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("cap,wgs,every", [(1, 1, 1), (1, 9, 2), (3, 65, 10), (16, 300, 7), (300, 256, 0)])
def test_units_come_back(hs, arena, kind, cap, wgs, every):
    print("sem", kind, cap, wgs, every, flush=True)
    sem = arena.sem_create(kind, 19, cap)
    storage = torch.arange(256 * 3, dtype=torch.float32, device="cuda")
    v = hs.sem_bench(arena, kind, sem, storage, wgs, 256, 2, 5, every)
    assert int(v[0].item()) == 0
    # a writer needs the whole capacity: one workgroup's writer gets it only if
    # every unit taken above was given back, and no writer is marked as waiting
    v = hs.sem_bench(arena, kind, sem, storage, 1, 256, 2, 2, 1)
    assert int(v[0].item()) == 0
    v = hs.sem_bench(arena, kind, sem, storage, 8, 256, 2, 2, 0)
    assert int(v[0].item()) == 0
