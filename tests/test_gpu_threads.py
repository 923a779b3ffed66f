"""Calls that wait for words the device leaves on the host, from several threads
on one map: each has words of its own and waits for its own stream."""
import threading
import time

import pytest
import torch

import workloads

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _together(count, work):
    """work(i) in `count` threads, each on a stream of its own; what they return."""
    torch.cuda.synchronize()
    out, gate = [None] * count, threading.Barrier(count)

    def body(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream(DEV)):
                gate.wait(30)
                out[i] = work(i)
        except Exception as exc:  # handed to the test's own thread
            out[i] = exc

    threads = [threading.Thread(target=body, args=(i,)) for i in range(count)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for o in out:
        if isinstance(o, Exception):
            raise o
    return out


def test_counters_read_by_several_threads(gpu_ash):
    engine = gpu_ash.ASHEngine(3, 5000, DEV)
    engine.insert_keys(torch.arange(9000, dtype=torch.int32, device=DEV).view(-1, 3))

    def read(_):
        # (`status` asks the device every time; more threads than cores, so that one
        # may be away while the others read)
        seen = {(engine.backend.status()["size"], engine.backend.size()) for _ in range(60)}
        return seen

    assert _together(40, read) == [{(3000, 3000)}] * 40


@pytest.mark.parametrize("queued", ["", "behind a millisecond of work and more"])
def test_queued_counters_read_by_several_threads(gpu_ash, queued):
    """The read-back that a streaming insert queues, looked at by all at once."""
    keys = torch.arange(900_000, dtype=torch.int32, device=DEV).view(-1, 3)
    work = torch.randn(8192, 8192, device=DEV)
    for n in (300_000, 299_999, 250_001):
        table = gpu_ash.HashSet(3, 600_000, DEV)
        if queued:
            work = torch.tanh(work @ work)
        table.insert(keys[:n])
        assert _together(4, lambda _: table.size()) == [n] * 4
        assert bool(table.find(keys[:n]).all())


def test_a_streaming_insert_that_waits_leaves_the_core(gpu_ash):
    """Behind some hundredths of a second of work the waiting thread sleeps."""
    keys = torch.arange(900_000, dtype=torch.int32, device=DEV).view(-1, 3)
    table = gpu_ash.HashSet(3, 600_000, DEV)
    work = torch.randn(8192, 8192, device=DEV)
    torch.tanh(work @ work)
    torch.cuda.synchronize()
    for _ in range(12):
        work = torch.tanh(work @ work)
    wall, cpu = time.perf_counter(), time.thread_time()
    table.insert(keys)
    assert table.size() == 300_000
    wall, cpu = time.perf_counter() - wall, time.thread_time() - cpu
    assert wall > 0.02 and cpu < 0.5 * wall, (wall, cpu)


def test_rays_sampled_by_several_threads(gpu_ash):
    grid, radii, centres = workloads.build_grid(gpu_ash, 800, 1, sparse_grid_dim=32, device=DEV)
    g = torch.Generator().manual_seed(5)
    rays = []
    for i in range(4):
        o = (torch.rand(500 + 37 * i, 3, generator=g) * 0.8 + 0.1).to(DEV)
        d = torch.randn(o.shape, generator=g).to(DEV)
        rays.append((o, d / d.norm(dim=1, keepdim=True)))

    def sample(i):
        near, far = grid.ray_find_near_far(*rays[i], 0.0, 2.0, 4 * grid.cell_size)
        return grid.ray_sample(*rays[i], near, far, 32)

    want = [sample(i) for i in range(4)]
    for _ in range(10):
        got = _together(4, sample)
        for a, b in zip(got, want):
            assert all(torch.equal(x, y) for x, y in zip(a, b))
