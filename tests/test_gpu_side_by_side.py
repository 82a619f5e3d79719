"""Two persistent launches at once on one GPU: on two streams with an arena each, and
beside a serving loop of the default size."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Work:
    """One kind of launch with its inputs and buffers: enqueue() on a stream, check()."""
    wgs = 0  # of a search: the default grid

    def __init__(self, hs, name):
        import torch
        import hsync.graph as G
        self.hs, self.name, self.arena = hs, name, hs.Arena()
        if name in ("bfs", "sssp", "pagerank"):
            row, col = G.rmat_csr(18 if name == "pagerank" else 14, 16, 5)
            self.g = G.Graph(row, col, G.weights(col.size, 5))
            self.src = int(np.argmax(np.diff(row.astype(np.int64))))
            self.out = torch.empty(self.g.n, dtype=torch.float32 if name == "pagerank" else torch.int32, device="cuda")
            self.work = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")
        elif name == "batch":
            lens = np.exp2(np.random.default_rng(4).uniform(0, 21, 90)).astype(np.int64)
            self.off = np.concatenate([[3], 3 + np.cumsum(np.concatenate([lens, [7 << 22]]))]).astype(np.uint64)
            self.x = torch.empty(int(self.off[-1]), dtype=torch.int32, device="cuda")
            hs.gen_uniform_u32(self.x, 7, 0, 2**32 - 1)
            self.out = torch.zeros_like(self.x)
        else:
            n = 9_000_001  # more than a round of half the CUs' registers
            self.x = torch.empty(n, dtype=torch.int32, device="cuda")
            hs.gen_uniform_u32(self.x, 6, 0, 2**32 - 1)
            self.out = torch.empty_like(self.x)
            self.scratch = torch.empty(8192, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()

    def enqueue(self, stream):
        import torch
        import hsync.graph as G
        with torch.cuda.stream(stream):  # a call's own tensors belong to its stream
            if self.name == "bfs":
                G.bfs(self.arena, self.g, self.src, num_wgs=self.wgs, level=self.out, work=self.work, sync=False)
            elif self.name == "sssp":
                G.sssp(self.arena, self.g, self.src, num_wgs=self.wgs, dist=self.out, work=self.work, sync=False)
            elif self.name == "pagerank":
                G.pagerank(self.arena, self.g, rank=self.out, work=self.work, sync=False)
            elif self.name == "batch":
                self.hs.scan_batch_u32(self.x, self.off, out=self.out, sync=False)
            else:
                self.hs.scan_u32(self.arena, self.x, out=self.out, scratch=self.scratch, sync=False)

    def check(self, stream, oracle):
        self.arena.sync(stream.cuda_stream)
        got = self.out.cpu().numpy()
        if self.name == "bfs":
            assert np.array_equal(got, oracle.bfs(self.g.h_row, self.g.h_col, self.src))
        elif self.name == "sssp":
            assert np.array_equal(got, oracle.sssp(self.g.h_row, self.g.h_col, self.g.h_w, self.src))
        elif self.name == "pagerank":
            want, _ = oracle.pagerank(self.g.h_row, self.g.h_col, alpha=0.85, tol=1e-6, max_iter=1000)
            assert float(np.abs(got - want).max()) < 1e-6
        elif self.name == "batch":
            stream.synchronize()
            x = oracle.gen_uniform_u32(7, got.size, 0, 2**32 - 1)
            for a, b in zip(self.off[:-1].astype(int), self.off[1:].astype(int)):
                assert np.array_equal(got[a:b].view(np.uint32), np.cumsum(x[a:b], dtype=np.uint32))
        else:
            x = oracle.gen_uniform_u32(6, got.size, 0, 2**32 - 1)
            assert np.array_equal(got.view(np.uint32), np.cumsum(x, dtype=np.uint32))

    def close(self):
        self.arena.close()


NAMES = ["bfs", "sssp", "scan", "batch", "pagerank"]


@pytest.mark.parametrize("a", NAMES)
@pytest.mark.parametrize("b", NAMES)
def test_on_two_streams(hs, oracle, a, b):
    import torch
    jobs = [Work(hs, a), Work(hs, b)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    try:
        for _ in range(10):
            for j, s in zip(jobs, streams):
                j.enqueue(s)
        for j, s in zip(jobs, streams):
            j.check(s, oracle)
    finally:
        for s in streams:
            s.synchronize()
        for j in jobs:
            j.close()


@pytest.mark.parametrize("names", [("bfs",) * 4, ("sssp",) * 4, ("bfs", "sssp", "bfs", "sssp")])
def test_four_searches_on_half_of_the_cus_each(hs, oracle, names):
    import torch
    jobs = [Work(hs, n) for n in names]
    streams = [torch.cuda.Stream() for _ in names]
    try:
        for j in jobs:
            j.wgs = hs.device_info()["num_cus"] // 2
        for _ in range(10):
            for j, s in zip(jobs, streams):
                j.enqueue(s)
        for j, s in zip(jobs, streams):
            j.check(s, oracle)
    finally:
        for s in streams:
            s.synchronize()
        for j in jobs:
            j.close()


def test_beside_the_serving_loop():
    """In a process of its own: HIP spreads a process's streams over four hardware
    queues, and a launch whose stream shares the queue of a kernel that does not end
    waits for it whatever room there is.  This one has two streams."""
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.split()[-1:] == ["done"], r.stdout + r.stderr[-2000:]


def _beside_the_serving_loop():
    """While the loop runs, nothing waits for the whole device: buffers and arenas are
    there before it starts, and a first call has made the allocations of a call."""
    import conftest  # noqa: F401  (the import paths)
    import torch
    import hsync as hs
    import oracle_lib
    from hsync.serve import Server
    oracle = oracle_lib.load()
    jobs = [Work(hs, name) for name in NAMES]
    s = torch.cuda.current_stream()
    for job in jobs:
        job.enqueue(s)
        job.check(s, oracle)
        job.out.zero_()
    x = torch.arange(5000, dtype=torch.int32, device="cuda")
    total = torch.zeros(1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    srv = Server()
    try:
        idx = srv.reduce(x, total)
        for job in jobs:
            print(job.name, flush=True)
            job.enqueue(s)
            job.check(s, oracle)
        assert srv.wait(idx)["status"] == 0
    finally:
        srv.stop()
    assert int(total.item()) == 5000 * 4999 // 2
    for job in jobs:
        job.close()
    print("done", flush=True)


if __name__ == "__main__":
    _beside_the_serving_loop()
