"""Rays that ask a map of the blocks in bounds, made by the call, against the
look-ups in the table: the same results, also for blocks outside the bounds and
after keys have come and gone."""
import ctypes
import os
import re

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("n", [8195, 66_000])   # eight and four lanes per ray in the march
@pytest.mark.parametrize("bounds", [(0, 31), (0, 28), (3, 17), (-5, 40), (7, 7), (-70, 91), (0, 161)])
def test_same_rays_with_and_without(gpu_ash, bounds, n):
    grid = gpu_ash.BoundedSparseDenseGrid(3, 6000, 1, 8, 32, device=DEV)
    backend, table = gpu_ash.grid.backend, grid.engine.backend
    g = torch.Generator().manual_seed(n + bounds[1])
    keys = torch.randint(0, 32, (7000, 3), generator=g).int().to(DEV)
    grid.engine.insert_keys(keys[:4000])
    grid.engine.insert_keys(torch.tensor([[2**31 - 1, 0, 4]], dtype=torch.int32, device=DEV))
    for sampling in (0, 1):   # (162 blocks an axis are too many)
        has_volume = backend.lib.ash_ray_volume_bytes(*bounds, n, sampling) > 0
        assert has_volume == (bounds[1] - bounds[0] < 161)
    o = (torch.rand(n, 3, generator=g) * 2.4 - 1.2).to(DEV)
    d = torch.nn.functional.normalize(torch.randn(n, 3, generator=g), dim=1).to(DEV)
    box = [torch.full((3,), x, device=DEV) for x in (-1.1, 1.1)]
    for turn in range(2):
        affine = grid._world_to_cell_affine(o)
        args = (table, o, d, *affine, *box, 0.0, 3.0 / grid.cell_size, 8.0)
        near, far = backend.ray_find_near_far_world(*args)
        for a, b in zip((near, far), backend.ray_find_near_far_world(*args, bounds)):
            assert torch.equal(a, b)
        args = (table, o, d, *affine, near, far, 64, 8.0)
        plain = backend.ray_sample_world(*args)
        for a, b in zip(plain, backend.ray_sample_world(*args, bounds)):
            assert torch.equal(a, b)
        assert len(plain[0]) > n
        grid.engine.erase(keys[1000:3000])
        grid.engine.insert_keys(keys[4000:])


@pytest.mark.parametrize("n", [8195, 66_000])
@pytest.mark.parametrize("far_block", [None, (40, 3, 5), (2**31 - 1, 0, 4)])
def test_rays_that_leave_the_volume(gpu_ash, far_block, n):
    """Ranges far beyond the grid (of rays that meet nothing), rays that are not finite,
    and the word that says whether a block is stored out there: all in bounds, one
    beyond them in the table, one in the second region."""
    grid = gpu_ash.BoundedSparseDenseGrid(3, 3000, 1, 8, 32, device=DEV)
    backend, table = gpu_ash.grid.backend, grid.engine.backend
    g = torch.Generator().manual_seed(n)
    grid.engine.insert_keys(torch.randint(0, 32, (2500, 3), generator=g).int().to(DEV))
    if far_block is not None:
        grid.engine.insert_keys(torch.tensor([far_block], dtype=torch.int32, device=DEV))
    o = torch.rand(n, 3, generator=g) * 256
    d = torch.nn.functional.normalize(torch.randn(n, 3, generator=g), dim=1)
    target = torch.tensor([40.0, 3, 5]) * 8 + 4
    d[::3] = torch.nn.functional.normalize(target - o[::3], dim=1)
    nan, inf = float("nan"), float("inf")
    d[:6] = torch.tensor([[0, 0, 0], [nan, 0, 1], [inf, 0, 1], [0, -inf, 0], [1e-3, 0, 0], [3e38, 0, -3e38]])
    o[6:9] = torch.tensor([[nan, 1, 1], [-inf, 1, 1], [1, 3e38, 1]])
    o, d = o.to(DEV), d.to(DEV)
    near = torch.where(torch.arange(n) % 2 == 0, -1.0, 20.0).to(DEV)
    far = torch.where(torch.arange(n) % 5 == 0, 60.0, 2000.0).to(DEV)
    near[9], far[10], near[11], far[12] = nan, nan, -inf, inf
    wide = [torch.full((3,), x, device=DEV) for x in (-inf, inf)]
    for box in ([torch.zeros(3, device=DEV), torch.full((3,), 256.0, device=DEV)], wide):
        args = (table, o, d, None, 1.0, *box, 0.0, 800.0, 8.0)
        for a, b in zip(backend.ray_find_near_far_world(*args), backend.ray_find_near_far_world(*args, (0, 31))):
            assert torch.equal(a, b)
    args = (table, o, d, None, 1.0, near, far, 128, 8.0)
    plain = backend.ray_sample_world(*args)
    for a, b in zip(plain, backend.ray_sample_world(*args, (0, 31))):
        assert a.dtype == b.dtype and torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))
    assert len(plain[0]) > n // 2   # (a block in thirteen is stored)


@pytest.mark.parametrize("zeros", [1, 2])
@pytest.mark.parametrize("n", [8195, 66_000])
def test_rays_along_axes(gpu_ash, zeros, n):
    """Directions with components of +0 and -0, from inside the bounds and from their faces."""
    grid = gpu_ash.BoundedSparseDenseGrid(3, 3000, 1, 8, 32, device=DEV)
    backend, table = gpu_ash.grid.backend, grid.engine.backend
    g = torch.Generator().manual_seed(n + zeros)
    grid.engine.insert_keys(torch.randint(0, 32, (2500, 3), generator=g).int().to(DEV))
    o = torch.rand(n, 3, generator=g) * 256
    d = torch.randn(n, 3, generator=g)
    axis = torch.randint(3, (n,), generator=g)
    for k in range(zeros):
        sign = torch.where(torch.rand(n, generator=g) < 0.5, 0.0, -0.0)
        d[torch.arange(n), (axis + k) % 3] = sign
        o[k::7, 0], o[k + 2::7, 1] = 0.0, 256.0
    o, d = o.to(DEV), torch.nn.functional.normalize(d, dim=1).to(DEV)
    box = [torch.full((3,), x, device=DEV) for x in (0.0, 256.0)]
    args = (table, o, d, None, 1.0, *box, 0.0, 800.0, 8.0)
    near, far = backend.ray_find_near_far_world(*args)
    for a, b in zip((near, far), backend.ray_find_near_far_world(*args, (0, 31))):
        assert torch.equal(a, b)
    # (a block in thirteen is stored, of the sixteen that a ray along an axis passes; a
    # ray that leaves at once from a face passes none)
    assert int((near >= 0).sum()) > n // 4


@pytest.mark.parametrize("n,where", [(8195, "one stream"), (8195, "two streams"), (8195, "captured"),
                                     (1024, "one stream"), (2048, "one stream")])
def test_blocks_of_earlier_calls_are_not_met(gpu_ash, n, where):
    """The volumes that are kept, of two sizes, marked with another number by every call:
    blocks come and go in between."""
    grid = gpu_ash.BoundedSparseDenseGrid(3, 3000, 1, 8, 32, device=DEV)
    backend, table = gpu_ash.grid.backend, grid.engine.backend
    g = torch.Generator().manual_seed(5)
    keys = torch.randint(0, 32, (2000, 3), generator=g).int().to(DEV)
    few_rays = backend.lib.ash_map_ray_volume_bytes
    assert few_rays(table._address, 0, 31, n, 0) > 0 and few_rays(table._address, 0, 31, 1023, 0) == 0
    o = (torch.rand(n, 3, generator=g) * 256).to(DEV)
    d = torch.nn.functional.normalize(torch.randn(n, 3, generator=g), dim=1).to(DEV)
    box = [torch.full((3,), x, device=DEV) for x in (0.0, 256.0)]
    args = (table, o, d, None, 1.0, *box, 0.0, 800.0, 8.0)
    streams = [torch.cuda.current_stream(), torch.cuda.Stream()]
    graph = torch.cuda.CUDAGraph()
    if where == "captured":
        grid.engine.insert_keys(keys)   # (a replay lists the blocks as the captured call did)
        grid.engine.erase(keys)
        backend.ray_find_near_far_world(*args, (0, 31))
        with torch.cuda.graph(graph):
            held = backend.ray_find_near_far_world(*args, (0, 31))
    for turn in range(300):
        few = keys[turn * 7 % 1900:][:100]
        if turn % 2 == 0:
            grid.engine.insert_keys(few)
        plain = backend.ray_find_near_far_world(*args)
        torch.cuda.synchronize()
        if where == "captured" and turn % 3 == 0:
            graph.replay()
            got = held
        else:
            with torch.cuda.stream(streams[turn % 2 if where == "two streams" else 0]):
                bounds = (0, 31) if turn % 5 else (0, 20)
                got = backend.ray_find_near_far_world(*args, bounds)
                if turn % 50 < 3:
                    samples = backend.ray_sample_world(table, o, d, None, 1.0, *got, 64, 8.0, bounds)
                    for a, b in zip(backend.ray_sample_world(table, o, d, None, 1.0, *got, 64, 8.0), samples):
                        assert torch.equal(a, b)
        torch.cuda.synchronize()
        for a, b in zip(plain, got):
            assert torch.equal(a, b), turn
        if turn % 2 == 1:
            grid.engine.erase(few)


def test_a_ray_beside_one_that_has_ended(gpu_ash):
    """The last lane of a ray that has ended stands in the block that the next ray's first
    lane asks the table about: it has not asked, and has no answer to give."""
    n, samples = 8193, 62
    grid = gpu_ash.BoundedSparseDenseGrid(3, 3000, 1, 8, 32, device=DEV)
    backend, table = gpu_ash.grid.backend, grid.engine.backend
    g = torch.Generator().manual_seed(n + samples)
    grid.engine.insert_keys(torch.randint(9, 23, (2500, 3), generator=g).int().to(DEV))
    o = (torch.rand(n, 3, generator=g) * 256).to(DEV)
    d = torch.nn.functional.normalize(torch.randn(n, 3, generator=g), dim=1).to(DEV)
    near, far = torch.zeros(n, device=DEV), (torch.rand(n, generator=g) * 200).to(DEV)
    args = (table, o, d, None, 1.0, near, far, samples, 8.0)
    for a, b in zip(backend.ray_sample_world(*args), backend.ray_sample_world(*args, (0, 31))):
        assert torch.equal(a, b)
    alone = [len(backend.ray_sample_world(table, o[r:r + 1], d[r:r + 1], None, 1.0, near[r:r + 1], far[r:r + 1],
                                          samples, 8.0)[0]) for r in range(4240, 4248)]
    counts = torch.bincount(backend.ray_sample_world(*args)[0], minlength=n)
    assert counts[4240:4248].tolist() == alone


@pytest.mark.parametrize("streams", [1, 2])
def test_numbers_come_again(gpu_ash, streams):
    """More than twice as many calls on every stream as there are numbers to mark with, with
    bounds of three sizes and origins that share a volume.  A call's blocks are stored for it
    alone, so that each keeps its number until this is given again; one beyond the narrower
    bounds comes and goes."""
    with open(os.path.join(os.path.dirname(__file__), os.pardir, "include", "ash_hip.h")) as f:
        marks = int(re.search(r"ASH_RAY_VOLUME_MARKS (\d+)", f.read())[1])
    grid = gpu_ash.BoundedSparseDenseGrid(3, 3000, 1, 8, 32, device=DEV)
    backend, table = gpu_ash.grid.backend, grid.engine.backend
    n, samples, each = 2048, 64, 30
    sizes = {backend.lib.ash_map_ray_volume_bytes(table._address, lo, hi, n, kind)
             for lo, hi in ((0, 31), (1, 30), (0, 28)) for kind in (0, samples)}
    assert len(sizes) == 1 and sizes.pop() > 0
    g = torch.Generator().manual_seed(streams)
    cube = torch.randperm(31 ** 3, generator=g)
    blocks = torch.stack([cube // 961, cube // 31 % 31, cube % 31], 1).int().to(DEV)
    beyond = torch.tensor([[31, 31, 31]], dtype=torch.int32, device=DEV)
    o = (torch.rand(n, 3, generator=g) * 256).to(DEV)
    d = torch.nn.functional.normalize(torch.randn(n, 3, generator=g), dim=1).to(DEV)
    box = [torch.full((3,), x, device=DEV) for x in (0.0, 256.0)]
    args = (table, o, d, None, 1.0, *box, 0.0, 800.0, 8.0)
    on = [torch.cuda.Stream() for _ in range(streams)]
    calls, met, turn = [0] * streams, 0, 0
    while min(calls) < 2 * marks + 2:
        k = turn % streams
        here = blocks[turn * each % (len(blocks) - each):][:each]
        if turn // streams % 3 == 0:
            here = torch.cat([here, beyond])
        grid.engine.insert_keys(here)
        plain = backend.ray_find_near_far_world(*args)
        torch.cuda.synchronize()
        with torch.cuda.stream(on[k]):
            bounds = ((0, 31), (1, 30), (0, 28))[turn % 5 % 3]
            got = backend.ray_find_near_far_world(*args, bounds)
            calls[k] += 1
            if turn % 7 == 0:
                asked = (table, o, d, None, 1.0, *got, samples, 8.0)
                for a, b in zip(backend.ray_sample_world(*asked, bounds), backend.ray_sample_world(*asked)):
                    assert torch.equal(a, b), turn
                calls[k] += 1
        torch.cuda.synchronize()
        for a, b in zip(plain, got):
            assert torch.equal(a, b), turn
        met += int((got[0] >= 0).any())
        grid.engine.erase(here)
        turn += 1
    # (no block was stored twice while its number could come again)
    assert met > turn // 2 and (marks + 2) * streams * each < len(blocks)


@pytest.mark.parametrize("n", [4096, 8195])
def test_scratch_that_holds_anything(gpu_ash, n):
    """The functions that clear their scratch themselves."""
    grid = gpu_ash.BoundedSparseDenseGrid(3, 3000, 1, 8, 32, device=DEV)
    backend, table = gpu_ash.grid.backend, grid.engine.backend
    lib, ptr = backend.lib, ctypes.c_void_p
    g = torch.Generator().manual_seed(n)
    grid.engine.insert_keys(torch.randint(0, 32, (2500, 3), generator=g).int().to(DEV))
    o = (torch.rand(n, 3, generator=g) * 256).to(DEV)
    d = torch.nn.functional.normalize(torch.randn(n, 3, generator=g), dim=1).to(DEV)
    lo, hi = (torch.full((3,), x, device=DEV) for x in (0.0, 256.0))
    near, far = backend.ray_find_near_far_world(table, o, d, None, 1.0, lo, hi, 0.0, 800.0, 8.0)
    at = lambda t: ptr(t.data_ptr())
    stream = ptr(torch.cuda.current_stream().cuda_stream)

    def scratch(sampling):
        size = lib.ash_ray_volume_bytes(0, 31, n, sampling)
        return torch.randint(0, 256, (size,), generator=g).to(torch.uint8).to(DEV) if size else None

    for _ in range(2):
        bytes_, nears, fars = scratch(0), torch.empty(n, device=DEV), torch.empty(n, device=DEV)
        assert bytes_ is not None
        assert lib.ash_ray_find_near_far_world(table._address, at(bytes_), 0, 31, at(o), at(d), None, 1.0, at(lo),
                                               at(hi), n, 0.0, 800.0, 8.0, at(nears), at(fars), stream) == 0
        assert torch.equal(nears, near) and torch.equal(fars, far)
        bytes_, stride = scratch(1), 64
        assert (bytes_ is None) == (n < 8192)
        counts = torch.empty(n, dtype=torch.int64, device=DEV)
        groups = torch.empty(lib.ash_ray_sample_groups(n), 2, dtype=torch.int64, device=DEV)
        stage, out = torch.empty(n, stride, 2, device=DEV), (ctypes.c_int64 * 2)()
        assert lib.ash_ray_sample_march(table._address, at(bytes_) if bytes_ is not None else None, 0, 31, at(o), at(d),
                                        None, 1.0, at(near), at(far), 0.0, 0.0, n, 32, 8.0, at(counts), at(groups),
                                        at(stage), stride, out, stream) == 0
        rays, starts, ends, prefix = backend.ray_sample_world(table, o, d, None, 1.0, near, far, 32, 8.0)
        assert out[0] == len(rays) and out[1] <= stride
        got = (torch.empty_like(rays), torch.empty_like(starts), torch.empty_like(ends), torch.empty_like(prefix))
        assert lib.ash_ray_sample_place(at(counts), at(groups), at(stage), stride, n, 1.0, *map(at, got), stream) == 0
        for a, b in zip(got, (rays, starts, ends, prefix)):
            assert torch.equal(a, b)
