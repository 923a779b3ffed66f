"""ash_convolution_cube against the kernels that go by the per-cell tables
(ash_convolution_forward): the same taps in the same order, so bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _grid(gpu_ash, channels, blocks, seed):
    grid = gpu_ash.SparseDenseGrid(3, blocks + 9, channels, 8, device=DEV)
    g = torch.Generator().manual_seed(seed)
    # a clump (inner blocks have all neighbours) and loners
    keys = torch.unique(torch.randint(0, 5, (3 * blocks, 3), generator=g), dim=0)[: max(1, blocks - 5)]
    keys = torch.cat([keys, torch.tensor([[50, 0, 0], [0, 50, 0], [0, 51, 1], [-7, 0, 3]])])[:blocks]
    grid.engine.insert_keys(keys.int().to(DEV))
    with torch.no_grad():
        grid.embeddings.copy_(torch.randn(grid.embeddings.shape, generator=g))
    return grid, g


@pytest.mark.parametrize("window", [3, 5, 7])
@pytest.mark.parametrize("channels", [1, 2, 3, 4, 5, 6, 7, 8])
def test_cube_equals_tables(gpu_ash, channels, window):
    backend = gpu_ash.grid.backend
    grid, g = _grid(gpu_ash, channels, 90, seed=channels * 10 + window)
    weights = torch.randn(window, window, window, channels, generator=g).to(DEV)
    c2g, c2c, lut = grid._window_tables(window // 2)
    _, listed = grid.engine.items()
    for rows in (listed, listed[::3].contiguous(), listed[:1], listed[:0]):
        got = backend.convolution_cube(grid.embeddings.data, weights, rows, lut, 8)
        want = backend.convolution_forward(
            grid.embeddings.data, weights.view(-1, channels),
            torch.ones(len(rows), 512, dtype=torch.bool, device=DEV), rows, grid.cell_indices, lut, c2c,
            c2g, 8)
        assert torch.equal(got, want)
    assert float(want.abs().sum()) == 0     # nothing listed: all rows cleared
    assert torch.equal(grid.convolution(grid.embeddings.data, weights),
                       backend.convolution_cube(grid.embeddings.data, weights, listed, lut, 8))


def test_sizes_left_to_the_other_kernels(gpu_ash):
    backend = gpu_ash.grid.backend
    supported = backend.lib.ash_convolution_cube_supported
    assert supported(262_143, 8, 3, 8, 0) and not supported(262_144, 8, 3, 8, 0)   # 4 GiB
    assert not supported(10, 4, 3, 4, 0) and not supported(10, 8, 9, 4, 0)
    assert not supported(10, 8, 3, 9, 0) and not supported(10, 8, 3, 4, 1)
    grid, g = _grid(gpu_ash, 9, 70, seed=1)
    out = grid.convolution(grid.embeddings.data, torch.randn(3, 3, 3, 9, generator=g).to(DEV))
    assert out.shape == grid.embeddings.shape and float(out.detach().abs().sum()) > 0


@pytest.mark.parametrize("channels,window", [(3, 3), (5, 3), (7, 3), (5, 5), (5, 7)])
def test_workgroups_that_walk_several_blocks(gpu_ash, channels, window):
    """More blocks than the device holds workgroups (at most seven a CU), an odd
    number of channels: wavefronts that only load and store go round as well."""
    blocks = 2003
    grid = gpu_ash.SparseDenseGrid(3, blocks + 9, channels, 8, device=DEV)
    g = torch.Generator().manual_seed(channels)
    keys = torch.unique(torch.randint(0, 16, (3 * blocks, 3), generator=g), dim=0)[:blocks]
    grid.engine.insert_keys(keys.int().to(DEV))
    weights = torch.randn(window, window, window, channels, generator=g).to(DEV)
    with torch.no_grad():
        grid.embeddings.copy_(torch.randn(grid.embeddings.shape, generator=g))
    c2g, c2c, lut = grid._window_tables(window // 2)
    _, listed = grid.engine.items()
    want = gpu_ash.grid.backend.convolution_forward(
        grid.embeddings.data, weights.view(-1, channels), torch.ones(blocks, 512, dtype=torch.bool, device=DEV),
        listed, grid.cell_indices, lut, c2c, c2g, 8)
    assert torch.equal(gpu_ash.grid.backend.convolution_cube(grid.embeddings.data, weights, listed, lut, 8), want)


@pytest.mark.parametrize("blocks,channels,window", [(1, 8, 7), (3000, 5, 3), (700_000, 1, 3)])
def test_rows_of_unlisted_blocks_are_cleared(gpu_ash, blocks, channels, window):
    """Fewer blocks than a workgroup looks at, more than there are workgroups, and
    more flags than the workgroups look at in one round (at most 16 a CU of 128
    threads); the first, the last and some in between are listed."""
    backend = gpu_ash.grid.backend
    g = torch.Generator().manual_seed(blocks)
    inputs = torch.randn(blocks, 512, channels, device=DEV)
    weights = torch.randn(window, window, window, channels, generator=g).to(DEV)
    lut = torch.full((blocks, 27), -1, dtype=torch.int64, device=DEV)
    lut[:, 13] = torch.arange(blocks, device=DEV)
    some = torch.unique(torch.cat([torch.tensor([0, blocks - 1]), torch.randint(blocks, (blocks // 3,), generator=g)]))
    listed = some[torch.randperm(len(some), generator=g)].to(DEV)
    everywhere = backend.convolution_cube(inputs, weights, torch.arange(blocks, device=DEV), lut, 8)
    for rows in (listed, listed[:0]):
        torch.full_like(inputs, 7.0)     # the result's memory does not start as zeros
        got = backend.convolution_cube(inputs, weights, rows, lut, 8)
        want = torch.zeros_like(inputs)
        want[rows] = everywhere[rows]
        assert torch.equal(got, want)


@pytest.mark.parametrize("channels,window", [(1, 3), (3, 3), (5, 5), (8, 3), (8, 7)])
def test_tensors_of_almost_four_gib(gpu_ash, channels, window):
    """Rows at both ends of the largest tensors, at 2 GiB and on either side of it, each with
    neighbours among the others and missing ones, against the same blocks in a small tensor;
    all other rows hold what is no number."""
    backend = gpu_ash.grid.backend
    blocks = 0xFFFFFFFF // (2048 * channels)
    assert backend.lib.ash_convolution_cube_supported(blocks, 8, window, channels, 0)
    assert not backend.lib.ash_convolution_cube_supported(blocks + 1, 8, window, channels, 0)
    middle = (1 << 31) // (2048 * channels)
    g = torch.Generator().manual_seed(window * 10 + channels)
    apart = torch.randint(4, blocks - 4, (50,), generator=g)
    rows = torch.unique(torch.cat([torch.tensor([0, 1, 2, blocks - 3, blocks - 2, blocks - 1]),
                                   torch.arange(middle - 2, middle + 3), apart]))
    n = len(rows)
    few = torch.randn(n, 512, channels, generator=g).to(DEV)
    weights = torch.randn(window, window, window, channels, generator=g).to(DEV)
    near = torch.randint(n, (n, 27), generator=g)
    near[torch.rand(n, 27, generator=g) < 0.3] = -1
    near[:, 13] = torch.arange(n)
    lut = torch.full((blocks, 27), -1, dtype=torch.int64, device=DEV)
    lut[rows.to(DEV)] = torch.where(near >= 0, rows[near.clamp_min(0)], -1).to(DEV)
    inputs = torch.full((blocks, 512, channels), float("nan"), device=DEV)
    inputs[rows.to(DEV)] = few
    order = torch.randperm(n, generator=g)
    got = backend.convolution_cube(inputs, weights, rows[order].to(DEV), lut, 8)
    grid, _ = _grid(gpu_ash, channels, 20, seed=1)
    c2g, c2c, _ = grid._window_tables(window // 2)
    want = backend.convolution_forward(
        few, weights.view(-1, channels), torch.ones(n, 512, dtype=torch.bool, device=DEV),
        torch.arange(n, device=DEV), grid.cell_indices, near.to(DEV), c2c, c2g, 8)
    assert float(want.abs().max()) > 1.0 and torch.equal(got[rows.to(DEV)], want)
    got[rows.to(DEV)] = 0.0
    assert int(torch.count_nonzero(got)) == 0   # (what is no number counts)
