"""A pass that reaches the embeddings through the first- and the second-order
backward of the module's forward: one dense gradient made by the second and
added to by the first, and the cases in which the first must leave it alone."""
import pytest
import torch

import workloads

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _losses(grid, x, hook=None):
    xq = x.clone().requires_grad_(True)
    feats, _ = grid(xq, "smooth_step")
    if hook is not None:
        hook(feats.grad_fn)
    (gx,) = torch.autograd.grad(feats[:, 0].sum(), xq, create_graph=True)
    return xq, (feats**2).mean(), (gx.norm(dim=-1) - 1).abs().mean(), gx


@pytest.mark.parametrize("embedding_dim", [1, 4, 5])
def test_second_order_gradient_is_carried_through_the_forward_node(gpu_ash, embedding_dim, monkeypatch):
    grid, radii, centres = workloads.build_grid(gpu_ash, 500, embedding_dim, sparse_grid_dim=32, device=DEV)
    x = workloads.ray_queries(grid, radii, centres, num_rays=64, samples_per_ray=50)
    backend = gpu_ash.grid_query.backend
    onto, real = [], backend.query_backward_forward_onto
    monkeypatch.setattr(backend, "query_backward_forward_onto",
                        lambda g, *a, **k: (onto.append(g.data_ptr()), real(g, *a, **k))[1], raising=False)
    want = []
    for which in (1, 2):
        grid.embeddings.grad = None
        _losses(grid, x)[which].backward()
        want.append(grid.embeddings.grad)
    want = want[0] + want[1]
    assert onto == [] and float(want.abs().max()) > 0

    def check(what):
        assert torch.allclose(grid.embeddings.grad, want, rtol=1e-4, atol=1e-6 * float(want.abs().max())), what

    # the plain pass: one tensor, which becomes .grad without a copy
    grid.embeddings.grad = None
    xq, value, eikonal, _ = _losses(grid, x)
    (value + eikonal).backward()
    check("plain")
    assert onto == [grid.embeddings.grad.data_ptr()] and xq.grad is not None

    # whoever keeps the carried gradient finds it unchanged: a hook before the
    # forward node, a hook behind the second-order node, a view kept by one
    for place in ("before", "behind", "view"):
        kept = []
        keep = lambda grads: kept.extend((g.detach() if place == "view" else g, g.clone())
                                         for g in grads if g is not None and g.shape == grid.embeddings.shape)
        grid.embeddings.grad = None
        hook = (lambda node: node.register_prehook(lambda outs: keep(outs))) if place == "before" else None
        xq, value, eikonal, gx = _losses(grid, x, hook)
        if place != "before":
            node = gx.grad_fn
            while "QueryBackward" not in node.name():
                node = node.next_functions[0][0]
            node.register_hook(lambda ins, outs: keep(ins))
        (value + eikonal).backward()
        check(place)
        assert len(onto) == 1 and len(kept) == 1, place
        assert torch.equal(*kept[0]), place

    # only the positions are asked for: no dense gradient at all
    xq, value, eikonal, _ = _losses(grid, x)
    calls = []
    real_bb = backend.query_backward_backward
    monkeypatch.setattr(backend, "query_backward_backward",
                        lambda *a, **k: (calls.append(k), real_bb(*a, **k))[1], raising=False)
    torch.autograd.grad(value + eikonal, xq)
    assert gpu_ash.grid_query.LAST_GRADIENT_PATH == "skipped"
    assert all(k.get("need_embeddings") is False for k in calls)

    # while the backward is recorded, and a third contribution to the parameter
    xq, value, eikonal, _ = _losses(grid, x)
    (got,) = torch.autograd.grad(value + eikonal, grid.embeddings, create_graph=True)
    assert torch.allclose(got, want, rtol=1e-4, atol=1e-6 * float(want.abs().max()))
    grid.embeddings.grad = None
    xq, value, eikonal, _ = _losses(grid, x)
    (value + eikonal + 0.5 * (grid.embeddings**2).sum()).backward()
    want = want + grid.embeddings.detach()
    check("decay")


def test_zero_offset_gradients_are_the_callers_own(gpu_ash):
    """The second-order offset gradient is zeros that a caller may write to:
    a tensor per call, no element of which another call sees."""
    backend = gpu_ash.grid_query.backend
    emb = torch.randn(1, 8, 2, device="cuda")
    n = 5
    ops = [emb, torch.rand(n, 3, device="cuda"), torch.zeros(n, dtype=torch.int64, device="cuda"),
           torch.zeros(n, dtype=torch.int64, device="cuda"), torch.ones(n, dtype=torch.bool, device="cuda"),
           torch.zeros(1, 8, dtype=torch.int64, device="cuda"),
           torch.zeros(8, 8, dtype=torch.int64, device="cuda"),
           torch.zeros(8, 8, dtype=torch.int64, device="cuda")]
    u, z = torch.randn(n, 3, device="cuda"), torch.randn(n, 2, device="cuda")
    first = backend.query_backward_backward(None, u, z, *ops, 2, "linear")[2]
    first[0, 0] = 7.0
    first += 1.0
    second = backend.query_backward_backward(None, u, z, *ops, 2, "linear")[2]
    assert second.shape == (n, 3) and not second.any()
