"""Losses of the features and of their gradient taken backward one after the
other through one graph, in both orders: the second-order gradient leads through
the forward node, which must let the other loss's pass come before or after."""
import pytest
import torch


@pytest.fixture()
def fused_ash(cpu_ash, oracle, monkeypatch):
    """The module's fused forward on the oracle: `query` and the interpolation
    as the operands of one call."""
    def grid_forward(table, x, emb, lut_g, lut_c2c, lut_c2g, grid_dim, interpolation,
                     need_operands=True, origin=None, cell_size=1.0):
        cells = (x if origin is None else x - origin) / cell_size
        grids, cell, offsets, masks = table.query_cells(cells, grid_dim)
        y = oracle.query_forward(emb, offsets, grids, cell, masks, lut_g, lut_c2c, lut_c2g,
                                 grid_dim, interpolation)
        return (y, masks, grids, cell, offsets) if need_operands else (y, masks, None, None, None)

    monkeypatch.setattr(oracle, "grid_forward", grid_forward, raising=False)
    return cpu_ash


def _grid(ash, device):
    grid = ash.BoundedSparseDenseGrid(3, 400, 3, grid_dim=4, sparse_grid_dim=16,
                                      bbox_min=torch.zeros(3), bbox_max=torch.ones(3), device=device)
    g = torch.Generator().manual_seed(3)
    x = (torch.rand(300, 3, generator=g) * 0.2 + 0.3).to(device)
    grid.spatial_init_(x, dilation=1, bidirectional=True)
    with torch.no_grad():
        grid.embeddings.copy_(torch.randn(grid.embeddings.shape, generator=g))
    table = grid.engine.backend
    if not hasattr(table, "query_cells"):
        table.query_cells = lambda cells, grid_dim: grid._query_elementwise(cells)
    return grid, x


def _losses(grid, x):
    xq = x.clone().requires_grad_(True)
    y, _ = grid(xq, "smooth_step")
    assert "FusedGridForward" in y.grad_fn.name()
    (gx,) = torch.autograd.grad(y[:, 0].sum(), xq, create_graph=True)
    return xq, (y**2).mean(), (gx.norm(dim=-1) - 1).abs().mean(), y


def _check(ash, grid, x):
    def added(*losses):
        with ash.dense_grad(grid):
            for loss in losses:
                loss.backward()

    ways = {
        "together": lambda a, b: (a + b).backward(),
        "value first": lambda a, b: (a.backward(), b.backward()),
        "gradient first": lambda a, b: (b.backward(), a.backward()),
        "value retained": lambda a, b: (a.backward(retain_graph=True), b.backward()),
        "gradient retained": lambda a, b: (b.backward(retain_graph=True), a.backward()),
        "added to .grad": lambda a, b: added(b, a),
    }
    want = None
    for name, way in ways.items():
        grid.embeddings.grad = None
        xq, value, eikonal, _ = _losses(grid, x)
        way(value, eikonal)
        got = grid.embeddings.grad, xq.grad
        want = want or got
        # float32 sums in another order
        assert all(torch.allclose(g, w, rtol=1e-5, atol=1e-6 * float(w.abs().max()))
                   for g, w in zip(got, want)), name

    # the value pass may come again as long as its graph is kept, and no longer,
    # also when a pass of the other loss has been there before
    for before in (False, True):
        xq, value, eikonal, y = _losses(grid, x)
        if before:
            eikonal.backward()
        grid.embeddings.grad = None
        value.backward(retain_graph=True)
        once = grid.embeddings.grad.clone()
        # (recorded from here: the same second-order gradient)
        (gx,) = torch.autograd.grad(y[:, 0].sum(), xq, create_graph=True)
        (gx.norm(dim=-1) - 1).abs().mean().backward(retain_graph=True)
        value.backward()
        assert torch.allclose(grid.embeddings.grad, want[0] + once, rtol=1e-5,
                              atol=1e-6 * float(want[0].abs().max())), before
        with pytest.raises(RuntimeError, match="second time"):
            value.backward()

    # the operands are checked for having been written to, before and after
    for before in (False, True):
        xq, value, eikonal, _ = _losses(grid, x)
        if before:
            eikonal.backward()
        with torch.no_grad():
            grid.embeddings.mul_(1.0)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            value.backward()


@pytest.mark.parametrize("arrived", [False, True])
def test_put_off_parts_are_added_to_one_tensor(cpu_ash, monkeypatch, arrived):
    """Several contributions that a second-order node has put off: one tensor takes
    them all, copied or made once, and what somebody else holds stays as it is."""
    gq = cpu_ash.grid_query
    targets = []
    monkeypatch.setattr(gq.backend, "query_backward_backward_onto",
                        lambda target, *rest: (targets.append(target), target.add_(1.0)), raising=False)
    embeddings, own = torch.randn(5, 8, 2), torch.zeros(5, 8, 2)
    carried = torch.randint(9, (5, 8, 2)).float() if arrived else None
    kept = carried.clone() if arrived else torch.zeros(5, 8, 2)
    somebody = [carried]   # (more than a node and what it calls hold of a gradient)
    parts = [((None, None), (embeddings,), target) for target in (None, own, None, None)]
    got = gq.add_put_off(parts, carried, 2, "linear")
    assert torch.equal(got, kept + 3) and torch.equal(own, torch.ones(5, 8, 2))
    assert not arrived or torch.equal(somebody[0], kept)
    assert {t.data_ptr() for t in targets} == {got.data_ptr(), own.data_ptr()}


def test_passes_one_after_the_other(fused_ash):
    _check(fused_ash, *_grid(fused_ash, torch.device("cpu")))


@pytest.mark.gpu
def test_passes_one_after_the_other_on_the_device(gpu_ash):
    _check(gpu_ash, *_grid(gpu_ash, torch.device("cuda:0")))
