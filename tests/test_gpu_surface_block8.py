"""ash_surface_block8_* against the kernels that go by the per-cell tables
(ash_marching_cubes_*, which the oracle checks): the same mesh, number for
number, and the module's transform bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _grid(gpu_ash, blocks, bounded, seed):
    if bounded:
        grid = gpu_ash.BoundedSparseDenseGrid(
            3, blocks + 5, 1, 8, 64, torch.tensor([-0.3, 0.1, 2.0]), torch.tensor([1.7, 1.2, 4.0]), DEV)
    else:
        grid = gpu_ash.UnBoundedSparseDenseGrid(3, blocks + 5, 1, 8, cell_size=0.013, device=DEV)
    g = torch.Generator().manual_seed(seed)
    # a clump with holes (blocks with all neighbours, and with any of them missing)
    edge = max(2, round((1.6 * blocks) ** (1 / 3)))
    keys = torch.unique(torch.randint(0, edge, (4 * blocks, 3), generator=g), dim=0)
    keys = keys[torch.randperm(len(keys), generator=g)[:blocks]]
    grid.engine.insert_keys(keys.int().to(DEV))
    grid.construct_grid_neighbor_lut_(radius=1, bidirectional=False)
    return grid, g


@pytest.mark.parametrize("blocks,stride,dtype,bounded", [
    (1, 1, torch.float32, True), (3, 5, torch.float32, False), (64, 64, torch.float64, True),
    (65, 2, torch.float64, False), (700, 5, torch.float32, True), (9000, 1, torch.float32, False),
    (700, 65, torch.float32, True),
])
def test_same_mesh_as_the_tables(gpu_ash, blocks, stride, dtype, bounded):
    grid, g = _grid(gpu_ash, blocks, bounded, seed=blocks + stride)
    rows = torch.randn(grid.num_embeddings, 512, stride, generator=g, dtype=dtype).to(DEV)
    # a tenth of the cells weigh too little
    rows[..., -1] = (torch.rand(rows.shape[:2], generator=g) * 10).to(DEV, dtype)
    sdf, weights = rows[..., 0], rows[..., -1]
    for iso, thr in ((0.1, 1.0), (50.0, 0.0), (0.0, 99.0)):   # the last two: nothing crossed, nothing heavy
        triangles, vertices = grid.surface_mesh(sdf, weights, iso, thr)
        _, listed = grid._blocks_in_spatial_order()
        want, points = gpu_ash.grid.backend.marching_cubes(
            sdf, weights, listed, grid.grid_coords, grid.lut_grid_nb2grid_idx, grid.cell_coords,
            grid.lut_cell_nb2cell_idx, grid.lut_cell_nb2grid_nb, 8, iso, thr)
        assert torch.equal(triangles, want) and triangles.dtype == want.dtype
        assert torch.equal(vertices, grid.transform_cell_to_world(points))
        if iso == 0.1 and stride > 1:
            assert len(want) > 10 * (blocks - 1)
    grid.transform_cell_to_world = lambda x: x + 1.0   # a caller's own
    assert torch.equal(grid.surface_mesh(sdf, weights, 0.1)[1],
                       gpu_ash.grid.backend.marching_cubes(
                           sdf, weights, listed, grid.grid_coords, grid.lut_grid_nb2grid_idx,
                           grid.cell_coords, grid.lut_cell_nb2cell_idx, grid.lut_cell_nb2grid_nb, 8,
                           0.1, 1.0)[1] + 1.0)


@pytest.mark.parametrize("stride,sdf,weight", [(2, 1, 0), (3, 0, 2), (4, 0, 1), (4, 3, 0), (5, 4, 0), (5, 1, 3),
                                               (6, 0, 5), (7, 0, 3), (8, 0, 7), (8, 4, 7), (9, 0, 8)])
def test_channels_anywhere_in_their_rows(gpu_ash, stride, sdf, weight):
    """Field and weights as channels of rows of two to eight (and nine) floats,
    the first of them 16-byte aligned or not, rows that nobody lists among them."""
    grid, g = _grid(gpu_ash, 150, False, seed=stride)
    rows = torch.randn(grid.num_embeddings, 512, stride, generator=g).to(DEV)
    rows[..., weight] = (torch.rand(rows.shape[:2], generator=g) * 10).to(DEV)
    f, w = rows[..., sdf], rows[..., weight]
    triangles, vertices = grid.surface_mesh(f, w, 0.1, 1.0)
    apart = grid.surface_mesh(f.contiguous(), w.contiguous(), 0.1, 1.0)
    assert len(triangles) > 1000
    assert torch.equal(triangles, apart[0]) and torch.equal(vertices, apart[1])


@pytest.mark.parametrize("light", [0.0, 0.03, 0.12, 0.2, 0.4])   # of the cells weigh too little
@pytest.mark.parametrize("field", ["checkerboard", "noise"])
def test_any_number_of_crossed_cells_in_a_block(gpu_ash, field, light):
    """Triangles are listed 192 crossed cells at a time, 64 a turn: from every
    cell of a block (light = 0 inside the clump) down to a few."""
    grid, g = _grid(gpu_ash, 300, False, seed=11)
    if field == "checkerboard":   # four triangles a cell, the most its code asks for
        c = torch.arange(8)
        sign = 1.0 - 2.0 * ((c.view(8, 1, 1) + c.view(1, 8, 1) + c.view(1, 1, 8)) % 2)
        sdf = sign.reshape(1, 512).repeat(grid.num_embeddings, 1).to(DEV)
    else:
        sdf = torch.randn(grid.num_embeddings, 512, generator=g).to(DEV)
    weights = (torch.rand(sdf.shape, generator=g) >= light).float().to(DEV)
    triangles, vertices = grid.surface_mesh(sdf, weights, 0.0, 0.5)
    _, listed = grid._blocks_in_spatial_order()
    want, points = gpu_ash.grid.backend.marching_cubes(
        sdf, weights, listed, grid.grid_coords, grid.lut_grid_nb2grid_idx, grid.cell_coords,
        grid.lut_cell_nb2cell_idx, grid.lut_cell_nb2grid_nb, 8, 0.0, 0.5)
    assert torch.equal(triangles, want) and torch.equal(vertices, grid.transform_cell_to_world(points))
    assert len(want) > 300


@pytest.mark.parametrize("blocks", [64, 700])
def test_rows_listed_before_and_not_now(gpu_ash, blocks):
    """The workspace is not cleared and comes back from call to call: rows of blocks that
    have gone, whose places of the call before name others now, or none."""
    grid, g = _grid(gpu_ash, blocks, True, seed=blocks)
    backend = gpu_ash.grid.backend
    rows = torch.randn(grid.num_embeddings, 512, 2, generator=g).to(DEV)
    for turn in range(6):
        grid.construct_grid_neighbor_lut_(radius=1, bidirectional=False)
        triangles, vertices = grid.surface_mesh(rows[..., 0], rows[..., 1], 0.1, -0.5)
        _, listed = grid._blocks_in_spatial_order()
        want, points = backend.marching_cubes(
            rows[..., 0], rows[..., 1], listed, grid.grid_coords, grid.lut_grid_nb2grid_idx, grid.cell_coords,
            grid.lut_cell_nb2cell_idx, grid.lut_cell_nb2grid_nb, 8, 0.1, -0.5)
        assert torch.equal(triangles, want) and torch.equal(vertices, grid.transform_cell_to_world(points))
        keys = grid.engine.items()[0]
        grid.engine.erase(keys[torch.randperm(len(keys), generator=g)[:len(keys) // 3].to(DEV)])
