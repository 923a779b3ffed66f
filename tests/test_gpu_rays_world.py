"""The ray methods of a grid (world units, transforms inside the kernels) against
the cell-unit functions on rays that torch has transformed: bit for bit."""
import pytest
import torch

import workloads

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.fixture(scope="module", params=["bounded", "unbounded"])
def scene(gpu_ash, request):
    grid, radii, centres = workloads.build_grid(gpu_ash, 3000, 2, 8, 64, device=DEV)
    if request.param == "unbounded":
        keys, _ = grid.engine.items()
        grid = gpu_ash.UnBoundedSparseDenseGrid(3, 3000, 2, 8, cell_size=0.0021, device=DEV)
        grid.engine.insert_keys(keys - 20)
    return grid


def _rays(grid, n, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    lo, hi = grid.get_bbox()
    keys, _ = grid.engine.items()
    target = grid.transform_cell_to_world((keys[torch.randint(len(keys), (n,), generator=g, device=DEV)] + 0.5)
                                          * grid.grid_dim)
    o = lo + (hi - lo) * torch.rand(n, 3, generator=g, device=DEV)
    d = target - o + 0.02 * torch.randn(n, 3, generator=g, device=DEV)
    return o, (d / d.norm(dim=1, keepdim=True).clamp_min(1e-6)).contiguous()


def _by_cell_units(grid, o, d, near, far, samples, t_max):
    cells, c, b = grid.transform_world_to_cell, grid.cell_size, grid.engine.backend
    lo, hi = (cells(x) for x in grid.get_bbox())
    from ash.grid import backend
    n, f = backend.ray_find_near_far(b, cells(o), d, lo, hi, 0.0, t_max / c, 1.0, float(grid.grid_dim))
    i, tn, tf, p = backend.ray_sample(b, cells(o), d, near / c, far / c, lo, hi, samples, float(grid.grid_dim))
    return n * c, f * c, i, tn * c, tf * c, p


# (70 000: one lane per ray; 4096 samples: more steps than a staging line holds)
@pytest.mark.parametrize("n,samples", [(0, 8), (1, 64), (31, 8), (33, 4096), (5000, 64), (70_000, 24)])
def test_world_rays_equal_transformed_rays(gpu_ash, scene, n, samples):
    o, d = _rays(scene, n, seed=n + 1)
    near, far = scene.ray_find_near_far(o, d, 0.0, 1.7, 0.01)
    got = scene.ray_sample(o, d, near, far, samples)
    want = _by_cell_units(scene, o, d, near, far, samples, 1.7)
    for a, b in zip((near, far, *got), want):
        assert a.dtype == b.dtype and torch.equal(a, b)
    if n > 1000:
        assert got[0].numel() > 5 * n and int((near >= 0).sum()) > n // 2
    # one range for all rays, given as numbers
    got = scene.ray_sample(o, d, 0.05, 0.9, samples)
    want = _by_cell_units(scene, o, d, torch.tensor(0.05, dtype=torch.float64), 0.9, samples, 1.7)[2:]
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_march_beyond_the_shared_chain_and_the_staging_line(gpu_ash, scene, monkeypatch):
    """More steps than a workgroup works out ahead, and rays with more samples
    than the staging area keeps."""
    o, d = _rays(scene, 300, seed=9)
    t_max = 4 * 1100 * scene.cell_size
    lo, hi = scene.get_bbox()
    # the box far away: rays start outside, so make it wide enough to march on
    grown = gpu_ash.grid.backend
    wide = (lo - 100, hi + 100)
    affine = scene._world_to_cell_affine(o)
    got = grown.ray_find_near_far_world(scene.engine.backend, o, d, *affine, *wide, 0.0,
                                        t_max / scene.cell_size, float(scene.grid_dim))
    cells, c = scene.transform_world_to_cell, scene.cell_size
    want = grown.ray_find_near_far(scene.engine.backend, cells(o), d, cells(wide[0]), cells(wide[1]), 0.0,
                                   t_max / c, 1.0, float(scene.grid_dim))
    assert torch.equal(got[0], want[0] * c) and torch.equal(got[1], want[1] * c)
    near, far = scene.ray_find_near_far(o, d, 0.0, 1.7, 0.01)
    plain = scene.ray_sample(o, d, near, far, 64)
    monkeypatch.setattr(gpu_ash.common, "RAY_STAGE_EXTRA", -60)
    for a, b in zip(plain, scene.ray_sample(o, d, near, far, 64)):
        assert torch.equal(a, b)
