"""ash_map_neighbors against the listing, find and scatter it replaces."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


class _WithoutTheKernel:
    """A map that offers what the general path asks for."""

    def __init__(self, backend):
        self.find, self.items = backend.find, backend.items


@pytest.mark.parametrize("radius,bidirectional", [(0, False), (1, False), (1, True), (2, True), (3, False)])
@pytest.mark.parametrize("blocks,far,erased", [(0, 0, 0), (1, 0, 0), (700, 0, 0), (700, 0, 300), (700, 60, 50)])
def test_same_table_as_the_general_path(gpu_ash, blocks, far, erased, radius, bidirectional):
    grid = gpu_ash.UnBoundedSparseDenseGrid(3, 901, 1, 2, device=DEV)
    g = torch.Generator().manual_seed(blocks + far)
    keys = torch.randint(-6, 6, (blocks, 3), generator=g).int()
    if far:   # beyond the packed range: kept in the general region, up to the end of int32
        keys[:far] += torch.tensor([2**31 - 7, 0, -2**31 + 6]).int()
    if blocks:
        grid.engine.insert_keys(keys.to(DEV))
    if erased:
        grid.engine.erase(keys[:erased].to(DEV))
        grid.engine.insert_keys(keys[: erased // 2].to(DEV))
    coords, lut = grid.construct_grid_neighbor_lut(radius, bidirectional)
    engine = grid.engine
    backend = engine.backend
    try:
        engine.backend = _WithoutTheKernel(backend)
        want_coords, want_lut = grid.construct_grid_neighbor_lut(radius, bidirectional)
    finally:
        engine.backend = backend
    assert coords.dtype == want_coords.dtype and lut.dtype == want_lut.dtype
    assert torch.equal(coords, want_coords) and torch.equal(lut, want_lut)
    assert int((lut[:, 0] >= 0).sum()) > 0 or radius > 0 or blocks == 0


@pytest.mark.parametrize("blocks", [31, 64, 700])   # 27 offsets: shares that end within a row, within and at a wavefront
def test_one_sided_window_of_three(gpu_ash, blocks):
    """The width of the two-sided window of one, from another first offset."""
    grid = gpu_ash.UnBoundedSparseDenseGrid(3, 901, 1, 2, device=DEV)
    g = torch.Generator().manual_seed(blocks)
    grid.engine.insert_keys(torch.randint(-6, 6, (blocks, 3), generator=g).int().to(DEV))
    coords, lut = grid.construct_grid_neighbor_lut(2, False)
    keys, indices = (t.cpu() for t in grid.engine.items())
    index = {tuple(k): int(i) for k, i in zip(keys.tolist(), indices)}
    coords, lut = coords.cpu(), lut.cpu()
    want = torch.full_like(lut, -1)
    for key, i in index.items():
        assert tuple(coords[i].tolist()) == key
        for n in range(27):
            there = tuple(key[d] + n // 3**d % 3 for d in range(3))
            want[i, n] = index.get(there, -1)
    assert torch.equal(lut, want)
