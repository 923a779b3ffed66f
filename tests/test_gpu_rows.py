"""The look-up with rows (ash_map_find_rows) and its transpose (ash_add_rows)
against torch's indexing on the indices that `find` returns: exact for the rows,
to the rounding of a reordered sum for the gradient."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _engine(gpu_ash, dim, stored, seed):
    g = torch.Generator().manual_seed(seed)
    keys = torch.unique(torch.randint(-90, 90, (2 * stored, dim), generator=g, dtype=torch.int32), dim=0)
    keys = keys[torch.randperm(len(keys), generator=g)][:stored]
    engine = gpu_ash.ASHEngine(dim, stored + 50, DEV)
    engine.insert_keys(keys.to(DEV))
    return engine, keys


def _queries(keys, n, seed):
    g = torch.Generator().manual_seed(seed)
    q = keys[torch.randint(len(keys), (n,), generator=g)].clone()
    q[torch.rand(n, generator=g) < 0.3, 0] += 1000
    if n > 2:
        q[1, 0] = 1 << 29     # does not fit the packed code of dims 3 and 4
    return q.to(DEV)


@pytest.mark.parametrize("dim", [1, 2, 3, 4])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 20_001])
def test_rows_are_those_of_the_found_indices(gpu_ash, dim, n):
    engine, keys = _engine(gpu_ash, dim, 100 if dim == 1 else 3000, seed=dim)
    q = _queries(keys, n, seed=n)
    indices, masks = engine.find(q)
    rows = engine.capacity
    tables = [torch.randn(rows, w, device=DEV) for w in (1, 3, 4, 67)]
    tables[1] = torch.randint(-9, 9, (rows, 3, 5), device=DEV)           # 120 bytes
    shifted = torch.randn(rows * 16 + 1, device=DEV)[1:].view(rows, 16)  # not 16-byte aligned
    backend = gpu_ash.core.backend
    for group in (tables, [shifted, torch.randn(rows, 8, device=DEV, dtype=torch.float64)]):
        assert backend.finds_rows_of(group, DEV)
        got_i, got_m, got = backend.find_rows(engine.backend, q, group)
        assert torch.equal(got_i, indices) and torch.equal(got_m, masks)
        for t, r in zip(group, got):
            assert torch.equal(r, t[indices])
        none, got_m, got = backend.find_rows(engine.backend, q, group, zero_misses=True, need_indices=False)
        assert none is None and torch.equal(got_m, masks)
        for t, r in zip(group, got):
            assert torch.equal(r, t[indices] * masks.view(-1, *[1] * (t.dim() - 1)).to(t.dtype))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("width,n", [(1, 1000), (3, 65), (16, 4097), (33, 300)])
def test_gradient_of_embedding_rows(gpu_ash, dtype, width, n):
    emb = gpu_ash.HashEmbedding(3, 701, width, DEV)
    emb.embedding = torch.nn.Parameter(torch.randn(701, width, device=DEV, dtype=dtype))
    g = torch.Generator().manual_seed(width)
    keys = torch.unique(torch.randint(-30, 30, (650, 3), generator=g, dtype=torch.int32), dim=0)
    emb.spatial_init_(keys.to(DEV))
    q = _queries(keys, n, seed=width + n)
    indices, masks = emb.engine.find(q)
    z = torch.randn(n, width, device=DEV, dtype=dtype, requires_grad=True)
    y = emb(q)
    assert torch.equal(y, emb.embedding[indices] * masks.unsqueeze(1))
    (got,) = torch.autograd.grad(y, emb.embedding, z, create_graph=True)
    terms = z.detach().double() * masks.unsqueeze(1)
    want = torch.zeros(701, width, device=DEV, dtype=torch.float64).index_add_(0, indices, terms)
    sums = torch.zeros_like(want).index_add_(0, indices, terms.abs())
    eps = 2.0**-24 if dtype == torch.float32 else 2.0**-53
    assert bool(((got.double() - want).abs() <= 16 * eps * sums).all())
    # and the gradient of the gradient: the look-up again
    u = torch.randn(701, width, device=DEV, dtype=dtype)
    (back,) = torch.autograd.grad(got, z, u)
    assert torch.equal(back, u[indices] * masks.unsqueeze(1))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_gradient_under_the_deterministic_flag(gpu_ash, dtype):
    """Rows that many keys share: the sums torch's backward of indexing takes,
    bit for bit, whichever pass the flag is first seen by."""
    emb = gpu_ash.HashEmbedding(3, 60, 8, DEV)
    emb.embedding = torch.nn.Parameter(torch.randn(60, 8, device=DEV, dtype=dtype))
    g = torch.Generator().manual_seed(2)
    keys = torch.unique(torch.randint(-30, 30, (50, 3), generator=g, dtype=torch.int32), dim=0)
    emb.spatial_init_(keys.to(DEV))
    q = _queries(keys, 50_001, seed=9)
    indices, masks = emb.engine.find(q)
    z = torch.randn(len(q), 8, generator=g, dtype=dtype).to(DEV)
    table = emb.embedding.detach().clone().requires_grad_(True)
    (masks.unsqueeze(-1) * table[indices]).backward(z)
    y = emb(q)
    try:
        torch.use_deterministic_algorithms(True)
        for out in (y, emb(q), emb(q)):
            (got,) = torch.autograd.grad(out, emb.embedding, z)
            assert torch.equal(got, table.grad)
        # and on to the gradient of the gradient
        zz = z.clone().requires_grad_(True)
        (got,) = torch.autograd.grad(emb(q), emb.embedding, zz, create_graph=True)
        u = torch.randn(60, 8, device=DEV, dtype=dtype)
        (back,) = torch.autograd.grad(got, zz, u)
    finally:
        torch.use_deterministic_algorithms(False)
    assert torch.equal(got, table.grad) and torch.equal(back, u[indices] * masks.unsqueeze(1))


def test_embedding_under_transforms_and_forward_mode(gpu_ash):
    """A batch of parameters (vmap) and a forward-mode tangent go through
    torch's own operations, as they always did."""
    emb = gpu_ash.HashEmbedding(3, 200, 4, DEV)
    g = torch.Generator().manual_seed(3)
    keys = torch.unique(torch.randint(-30, 30, (150, 3), generator=g, dtype=torch.int32), dim=0)
    emb.spatial_init_(keys.to(DEV))
    q = _queries(keys, 333, seed=4)
    indices, masks = emb.engine.find(q)

    def rows(table):
        return torch.func.functional_call(emb, {"embedding": table}, (q,))

    stack = torch.randn(3, 200, 4, device=DEV)
    want = stack[:, indices] * masks.view(1, -1, 1)
    assert torch.equal(torch.func.vmap(rows)(stack), want)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(stack[0], stack[1])
        value, tangent = torch.autograd.forward_ad.unpack_dual(rows(dual))
    assert torch.equal(value, want[0]) and torch.equal(tangent, want[1])


@pytest.mark.parametrize("dim,n,widths,alike", [
    (3, 1 << 21, (3, 1), False), (3, (1 << 21) + 1, (1, 4, 3), False), (1, (1 << 21) + 4095, (5, 1, 1, 1), False),
    (4, 2_500_001, (1, 4), False), (2, 1 << 21, (3, 3), True)])
def test_rows_of_large_batches_in_index_order(gpu_ash, dim, n, widths, alike):
    """Two million queries and more on two tables and more: rows are read in index
    order, and equal those that batches below the limit get key by key."""
    g = torch.Generator(device=DEV).manual_seed(dim)
    stored = 1_200_000
    keys = torch.randint(-(1 << 28 if dim == 1 else 9000), 1 << 28 if dim == 1 else 9000, (stored, dim), generator=g,
                         device=DEV, dtype=torch.int32)
    engine = gpu_ash.ASHEngine(dim, stored + 100_000, DEV)
    engine.insert_keys(keys)
    q = keys[torch.randint(stored, (n,), generator=g, device=DEV)]
    q[torch.rand(n, generator=g, device=DEV) < 0.3, 0] += 1 << 20 if dim < 4 else 20_000
    if alike:
        q[:] = keys[7]
    q[1, 0] = 1 << 29
    rows = engine.capacity
    # the last table ends before the stored indices do: zeros from there on
    tables = [torch.randint(1 << 30, (rows - (300_000 if v == len(widths) - 1 else 0), w), generator=g, device=DEV,
                            dtype=torch.int32) for v, w in enumerate(widths)]
    row_bytes, src_rows = ((ctypes.c_int64 * len(widths))(*each) for each in
                           ((4 * w for w in widths), (len(t) for t in tables)))
    assert gpu_ash.common.load_library().ash_map_find_rows_scratch_bytes(
        engine.backend._address, n, len(widths), row_bytes, src_rows) > 0
    for zero_misses in (False, True):
        got_i, got_m, got = gpu_ash.core.backend.find_rows(engine.backend, q, tables, zero_misses=zero_misses)
        parts = [gpu_ash.core.backend.find_rows(engine.backend, p, tables, zero_misses=zero_misses)
                 for p in q.split(500_000)]
        assert torch.equal(got_i, torch.cat([p[0] for p in parts]))
        assert torch.equal(got_m, torch.cat([p[1] for p in parts]))
        for v, r in enumerate(got):
            assert torch.equal(r, torch.cat([p[2][v] for p in parts]))
    none, got_m, again = gpu_ash.core.backend.find_rows(engine.backend, q, tables, zero_misses=True, need_indices=False)
    assert none is None and all(torch.equal(a, b) for a, b in zip(again, got))


@pytest.mark.parametrize("n", [2_400_257, 2_400_257 + 511])   # a last chunk of 1 and of 512 queries
@pytest.mark.parametrize("widths", [(1, 1), (2, 1), (3, 1), (1, 4), (3, 3), (4, 3), (1, 4, 3), (5, 1, 1, 1), (4, 4)])
def test_chunks_of_few_stored_keys_are_served_key_by_key(gpu_ash, widths, n):
    """Rows in index order, from one chunk of 4096 queries to the next: none, all and
    a share next to every bound (three, four, six and seven eighths) of the keys are
    stored."""
    g = torch.Generator(device=DEV).manual_seed(n)
    rows = 2_300_000
    at = torch.arange(rows, device=DEV)
    keys = torch.stack([at & 1023, (at >> 10) & 1023, at >> 20], 1).int()
    engine = gpu_ash.ASHEngine(3, rows, DEV)
    engine.insert_keys(keys)
    q = keys[torch.randint(rows, (n,), generator=g, device=DEV)]
    stored = torch.tensor([0, 1535, 1536, 2047, 2048, 3071, 3072, 3583, 3584, 4095, 4096], device=DEV)
    of = torch.arange(n, device=DEV)
    chunk, place = of // 4096, of % 4096
    q[(place * 1237 % 4096) >= stored[chunk % len(stored)], 0] += 4096
    tables = [torch.randint(1 << 30, (rows - (200_000 if v == len(widths) - 1 else 0), w), generator=g, device=DEV,
                            dtype=torch.int32) for v, w in enumerate(widths)]   # the last ends early: zeros from there on
    row_bytes, src_rows = ((ctypes.c_int64 * len(widths))(*each) for each in
                           ((4 * w for w in widths), (len(t) for t in tables)))
    assert gpu_ash.common.load_library().ash_map_find_rows_scratch_bytes(
        engine.backend._address, n, len(widths), row_bytes, src_rows) > 0
    for zero_misses in (False, True):
        got_i, got_m, got = gpu_ash.core.backend.find_rows(engine.backend, q, tables, zero_misses=zero_misses)
        parts = [gpu_ash.core.backend.find_rows(engine.backend, p, tables, zero_misses=zero_misses)
                 for p in q.split(500_000)]
        assert torch.equal(got_i, torch.cat([p[0] for p in parts]))
        assert torch.equal(got_m, torch.cat([p[1] for p in parts]))
        for v, r in enumerate(got):
            assert torch.equal(r, torch.cat([p[2][v] for p in parts]))


@pytest.mark.parametrize("widths,rows,queries", [   # the least number of queries, None: never
    ((1, 1), 12_000_000, 3_000_000), ((3, 1), 12_000_000, 3_000_000), ((3, 2), 12_000_000, 12_000_000),
    ((4, 4), 12_000_000, 12_000_000), ((3, 3), 41_000_000, 10_250_000), ((4, 4), 31_000_000, 15_500_000),
    ((3, 1), 4_000_000, 1 << 21), ((3, 1), 1_000_000, None), ((4, 5), 4_000_000, None), ((4,), 12_000_000, None)])
def test_which_batches_read_rows_in_index_order(gpu_ash, widths, rows, queries):
    engine = gpu_ash.ASHEngine(3, 100, DEV)
    row_bytes, src_rows = ((ctypes.c_int64 * len(widths))(*each) for each in
                           ((4 * w for w in widths), (rows for w in widths)))

    def scratch(n):
        return gpu_ash.common.load_library().ash_map_find_rows_scratch_bytes(
            engine.backend._address, n, len(widths), row_bytes, src_rows)

    assert scratch((queries or 100_000_000) - 1) == 0
    # an index and a place per query, its rows, and little beside them
    assert queries is None or 0 < scratch(queries) < queries * (7 + 4 * sum(widths))
