"""Rays that ask a map of the blocks in bounds, made by the call, against the
look-ups in the table: the same results, also for blocks outside the bounds and
after keys have come and gone."""
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
