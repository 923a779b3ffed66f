"""The embedding gradients of the first- and the second-order backward in one
pass over the queries: the kernels against the oracle, and the passes of the
engine in which the second-order node may and may not leave its share to the
forward node."""
import gc
import threading

import pytest
import torch

import workloads
from helpers import assert_close_sums
from test_gpu_query import _eps, _make_grid, _operands, _queries, _to_cpu, _tol

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


# 600 001 queries: tables of cells in LDS; blocks of 4^3 also the wide workgroups
@pytest.mark.parametrize("dtype,grid_dim,width,n", [
    (dtype, 4, width, n) for dtype in (torch.float32, torch.float64) for width in (1, 2, 3, 4, 5, 8, 16)
    for n in (1, 257)] + [(torch.float32, 4, 4, 600_001), (torch.float32, 8, 4, 600_001),
                          (torch.float32, 11, 4, 600_001), (torch.float32, 4, 5, 600_001),
                          (torch.float64, 4, 3, 600_001)])
@pytest.mark.parametrize("need_offsets", [True, False])
def test_both_orders_against_the_oracle(gpu_ash, oracle, dtype, grid_dim, width, n, need_offsets):
    grid = _make_grid(gpu_ash, grid_dim, width, 1, dtype=dtype, seed=width, holes=2)
    ops = _operands(grid, _queries(grid_dim, 1, n, seed=n, margin=1.0))
    g = torch.Generator().manual_seed(n)
    z, u, z2 = ((torch.rand(n, w, generator=g, dtype=dtype) - 0.5).to(DEV) for w in (width, 3, width))
    start = (torch.rand(ops[0].shape, generator=g, dtype=dtype) - 0.5).to(DEV)
    host = gpu_ash.grid_query.backend.host
    cpu = _to_cpu(ops)
    want, want_off = oracle.query_backward_forward(z.cpu(), *cpu, grid_dim, "smooth_step")
    want = want + oracle.query_backward_backward(None, u.cpu(), z2.cpu(), *cpu, grid_dim, "smooth_step")[1]
    sums = (oracle.query_term_sums(u, z, *cpu, grid_dim, "smooth_step")["bf_embeddings"]
            + oracle.query_term_sums(u, z2, *cpu, grid_dim, "smooth_step")["bb_embeddings"])
    bound = dict(eps=_eps(dtype), **_tol(dtype))
    got, got_off = host.query_backward_both(z, u, z2, list(ops), "smooth_step", need_offsets, None)
    assert_close_sums(got, want, sums, what="zeroed", **bound)
    acc, _ = host.query_backward_both(z, u, z2, list(ops), "smooth_step", need_offsets, start)
    assert acc.data_ptr() == start.data_ptr()
    began = acc.cpu().double() - got.cpu().double()   # what was there, up to the same rounding
    g = torch.Generator().manual_seed(n)
    for w in (width, 3, width):
        torch.rand(n, w, generator=g, dtype=dtype)
    first = torch.rand(ops[0].shape, generator=g, dtype=dtype) - 0.5
    assert_close_sums(began, first, 2 * sums + 2 * first.double().abs(), what="added", **bound)
    if need_offsets:
        assert torch.allclose(got_off.cpu(), want_off, **_tol(dtype))
    else:
        assert got_off is None


def test_rows_of_four_off_their_alignment(gpu_ash):
    """z of the second order at an address that is no multiple of 16."""
    grid = _make_grid(gpu_ash, 4, 4, 1, seed=3)
    ops = _operands(grid, _queries(4, 1, 1000, seed=4))
    z, u = torch.rand(1000, 4, device=DEV), torch.rand(1000, 3, device=DEV)
    z2 = torch.rand(4001, device=DEV)[1:].view(1000, 4)
    host = gpu_ash.grid_query.backend.host
    got, _ = host.query_backward_both(z, u, z2, list(ops), "linear", False, None)
    want, _ = host.query_backward_both(z, u, z2.clone(), list(ops), "linear", False, None)
    assert torch.allclose(got, want, rtol=1e-5, atol=1e-5)


class _Fails(torch.autograd.Function):
    armed = False

    @staticmethod
    def forward(ctx, y):
        return y.clone()

    @staticmethod
    def backward(ctx, z):
        if _Fails.armed:
            raise ValueError("on purpose")
        return z


@pytest.fixture()
def scene(gpu_ash, monkeypatch):
    grid, radii, centres = workloads.build_grid(gpu_ash, 300, 4, sparse_grid_dim=32, device=DEV)
    x = workloads.ray_queries(grid, radii, centres, num_rays=64, samples_per_ray=30)
    backend = gpu_ash.grid_query.backend
    put_off, real = [], backend.query_backward_backward
    monkeypatch.setattr(gpu_ash.grid_query, "PUT_OFF_FROM", 0)
    monkeypatch.setattr(backend, "query_backward_backward",
                        lambda *a, **k: (put_off.append(k.get("later", False)), real(*a, **k))[1], raising=False)
    return gpu_ash, grid, x, put_off


def _grad(grid, loss, **how):
    grid.embeddings.grad = None
    loss.backward(**how)
    return grid.embeddings.grad.clone()


def _close(got, want):
    return torch.allclose(got, want, rtol=1e-4, atol=1e-6 * float(want.abs().max()))


def _norm_loss(y, xq, channel):
    (gx,) = torch.autograd.grad(y[:, channel].sum(), xq, create_graph=True)
    return (gx.norm(dim=-1) - 1).abs().mean()


def _separately(grid, x, channels):
    total = 0
    for what in ("value", *channels):
        xq = x.clone().requires_grad_(True)
        y, _ = grid(xq, "smooth_step")
        total = total + _grad(grid, (y**2).mean() if what == "value" else _norm_loss(y, xq, what))
    return total


def test_several_second_order_nodes_of_one_forward(scene):
    ash, grid, x, put_off = scene
    want = _separately(grid, x, (0, 2, 3))
    for inside in (False, True):
        del put_off[:]
        xq = x.clone().requires_grad_(True)
        y, _ = grid(xq, "smooth_step")
        loss = (y**2).mean() + sum(_norm_loss(y, xq, c) for c in (0, 2, 3))
        grid.embeddings.grad = None
        if inside:
            with ash.dense_grad(grid):
                loss.backward()
        else:
            loss.backward()
        assert put_off == [True] * 3 and _close(grid.embeddings.grad, want)


def test_a_pass_that_fails_in_between_leaves_nothing_behind(scene):
    ash, grid, x, put_off = scene
    want = _separately(grid, x, (0,))
    xq = x.clone().requires_grad_(True)
    y, _ = grid(xq, "smooth_step")
    # nodes are run latest first, as each thread counts them: recorded in a thread
    # of its own, this one is run after the second-order node
    value = []
    thread = threading.Thread(target=lambda: value.append((_Fails.apply(y)**2).mean()))
    thread.start()
    thread.join()
    loss = value[0] + _norm_loss(y, xq, 0)
    _Fails.armed = True
    del put_off[:]
    try:
        with pytest.raises(ValueError, match="on purpose"):
            loss.backward(retain_graph=True)
    finally:
        _Fails.armed = False
    assert put_off == [True]
    assert _close(_grad(grid, loss, retain_graph=True), want) and _close(_grad(grid, loss), want)


def test_a_pass_that_fails_keeps_no_operands(scene):
    """... nor the memory of what it had put off, while the graph lives."""
    ash, grid, x, put_off = scene
    xq = x.clone().requires_grad_(True)
    y, _ = grid(xq, "smooth_step")
    value = []
    thread = threading.Thread(target=lambda: value.append((_Fails.apply(y)**2).mean()))
    thread.start()
    thread.join()
    loss = value[0] + _norm_loss(y, xq, 0)
    grid.embeddings.grad = None
    loss.backward(retain_graph=True)         # what a first pass leaves for good
    grid.embeddings.grad = None
    xq.grad = None
    gc.collect()
    before = torch.cuda.memory_allocated()
    _Fails.armed = True
    del put_off[:]
    try:
        for _ in range(3):
            try:
                loss.backward(retain_graph=True)
            except ValueError:
                pass
    finally:
        _Fails.armed = False
    gc.collect()
    assert put_off == [True] * 3 and torch.cuda.memory_allocated() == before


def test_putting_off_copies_nothing(gpu_ash):
    """Operands that are not contiguous are copied where they are used, not where
    they are put off."""
    grid = _make_grid(gpu_ash, 4, 4, 1, seed=3)
    ops = _operands(grid, _queries(4, 1, 100_000, seed=4))
    z, u = torch.ones(1, 4, device=DEV).expand(100_000, 4), torch.ones(1, 3, device=DEV).expand(100_000, 3)
    host = gpu_ash.grid_query.backend.host
    start = torch.zeros_like(ops[0])
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    got = host.query_gradient_later(u, z, list(ops), "linear", start)
    assert got.data_ptr() == start.data_ptr() and torch.cuda.max_memory_allocated() == before
    for wrong in ((u, z[:, :3]), (u[:-1], z), (u, z.double()), (u.cpu(), z)):
        with pytest.raises(RuntimeError):
            host.query_gradient_later(*wrong, list(ops), "linear", start)


def test_gradients_that_somebody_sees_are_whole(scene):
    ash, grid, x, put_off = scene
    xq = x.clone().requires_grad_(True)
    y, _ = grid(xq, "smooth_step")
    second = _grad(grid, _norm_loss(y, xq, 0))
    xq = x.clone().requires_grad_(True)
    y, _ = grid(xq, "smooth_step")
    seen = []
    y.grad_fn.register_prehook(lambda grads: seen.extend(g.clone() for g in grads
                                                         if g is not None and g.shape == second.shape))
    loss = (y**2).mean() + _norm_loss(y, xq, 0)
    del put_off[:]
    total = _grad(grid, loss)
    assert put_off == [False] and len(seen) == 1 and _close(seen[0], second)
    assert _close(total, _separately(grid, x, (0,)))


def test_a_gradient_recorded_under_another_stream(scene):
    ash, grid, x, put_off = scene
    want = _separately(grid, x, (0,))
    xq = x.clone().requires_grad_(True)
    y, _ = grid(xq, "smooth_step")
    value = (y**2).mean()
    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(other):
        norm = _norm_loss(y, xq, 0)
    torch.cuda.current_stream().wait_stream(other)
    del put_off[:]
    # (recorded on the forward's stream all the same)
    assert _close(_grad(grid, value + norm), want) and put_off == [True]


@pytest.mark.parametrize("more", [0, -1])
def test_few_queries_are_not_put_off(scene, monkeypatch, more):
    ash, grid, x, put_off = scene
    monkeypatch.setattr(ash.grid_query, "PUT_OFF_FROM", len(x) - more)
    want = _separately(grid, x, (0, 2))
    del put_off[:]
    xq = x.clone().requires_grad_(True)
    y, _ = grid(xq, "smooth_step")
    got = _grad(grid, (y**2).mean() + _norm_loss(y, xq, 0) + _norm_loss(y, xq, 2))
    assert put_off == [more == 0] * 2 and _close(got, want)


@pytest.mark.parametrize("dtype,width,n", [
    (dtype, width, n) for dtype in (torch.float32, torch.float64) for width in (1, 3, 4, 5, 16)
    for n in (1, 1000)] + [(torch.float32, 4, 600_001), (torch.float32, 5, 600_001)])
@pytest.mark.parametrize("cell_size", [0.015, 3.0])
def test_gradients_by_positions_in_units_of_a_cell(gpu_ash, dtype, width, n, cell_size):
    """The kernels multiply as torch divides: gradients with respect to the positions to
    the bit, those that the atomics add up to the rounding of their order."""
    grid = _make_grid(gpu_ash, 4, width, 1, dtype=dtype, seed=width, holes=2)
    ops = list(_operands(grid, _queries(4, 1, n, seed=n, margin=1.0)))
    g = torch.Generator().manual_seed(n)
    z, u, z2 = ((torch.rand(n, w, generator=g, dtype=dtype) - 0.5).to(DEV) for w in (width, 3, width))
    host = gpu_ash.grid_query.backend.host
    tol = dict(rtol=1e-5 if dtype == torch.float32 else 1e-12, atol=1e-5 * n ** 0.5)

    emb, off = host.query_backward_forward(z, ops, "smooth_step", True, True, None, cell_size)
    emb1, off1 = host.query_backward_forward(z, ops, "smooth_step", True, True, None)
    assert torch.equal(off, off1 / cell_size) and torch.allclose(emb, emb1, **tol)
    none, off = host.query_backward_forward(z, ops, "smooth_step", False, True, None, cell_size)
    assert none is None and torch.equal(off, off1 / cell_size)
    for need_z, need_emb in ((True, True), (True, False), (False, True)):
        gz, emb = host.query_backward_backward(u, z, ops, "linear", need_z, need_emb, None, cell_size)
        gz1, emb1 = host.query_backward_backward(u / cell_size, z, ops, "linear", need_z, need_emb, None)
        assert not need_z or torch.equal(gz, gz1)
        assert not need_emb or torch.allclose(emb, emb1, **tol)
    for need_off in (True, False):
        emb, off = host.query_backward_both(z, u, z2, ops, "smooth_step", need_off, None, cell_size)
        emb1, off1 = host.query_backward_both(z, u / cell_size, z2, ops, "smooth_step", need_off, None)
        assert torch.allclose(emb, emb1, **tol)
        assert not need_off or torch.equal(off, off1 / cell_size)
