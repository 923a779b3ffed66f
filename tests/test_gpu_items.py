"""Listings with their value rows: against torch's indexing by the listed indices, at the
edges of the rounds that a workgroup takes, for row widths copied along and not."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.fixture(scope="module")
def ash():
    import ash as module

    return module


def _keys(first, n, dim=3):
    i = torch.arange(first, first + n, dtype=torch.int32)
    k = torch.stack([i % 251, i // 251 % 257, i // (251 * 257), i % 7], dim=1)
    return (k[:, :dim] if dim > 1 else i.view(-1, 1)).contiguous().to(DEV)


def _check(hm, stored):
    keys, indices, rows = hm.items(return_values=True)
    assert keys.shape[0] == stored.shape[0] == torch.unique(indices).numel()
    found, masks = hm.engine.find(keys)
    assert bool(masks.all()) and torch.equal(found, indices)
    assert torch.equal(torch.unique(keys, dim=0), torch.unique(stored, dim=0))
    for name, got in rows.items():
        assert torch.equal(got, hm.values[name][indices]), name
    only = hm.items(return_indices=False, return_values=True)
    assert len(only) == 2 and only[0].shape == keys.shape


@pytest.mark.parametrize("dim", [1, 2, 3, 4])
@pytest.mark.parametrize("capacity", [1, 1023, 1025, 40_000])
def test_rows_of_a_listing(ash, dim, capacity):
    widths = {"a": 3, "b": 1, "c": 16, "d": 5}
    hm = ash.HashMap(dim, widths, capacity, DEV)
    for v in hm.values.values():
        v.uniform_()
    n = max(1, capacity * 2 // 3)
    dim_keys = _keys(0, n, dim) if dim != 2 else _keys(0, n, 3)[:, :2].contiguous()
    dim_keys = torch.unique(dim_keys, dim=0)
    hm.insert(dim_keys, {k: torch.rand(len(dim_keys), w, device=DEV) for k, w in widths.items()})
    _check(hm, dim_keys)                       # entry i under index i
    gone = dim_keys[: len(dim_keys) // 3]
    if len(gone):
        hm.erase(gone)
    for _ in range(18):                        # more listings than there are cursors
        _check(hm, dim_keys[len(gone):])


@pytest.mark.parametrize("capacity", [256 * 1024, 256 * 1024 + 1, 1024 * 1024, 1024 * 1024 + 1])
def test_listings_at_the_bounds_of_the_rounds(ash, capacity):
    hm = ash.HashMap(3, {"a": 3, "b": 1}, capacity, DEV)
    keys = _keys(0, capacity)
    hm.insert(keys, {"a": torch.rand(capacity, 3, device=DEV), "b": torch.rand(capacity, 1, device=DEV)})
    hm.erase(keys[5::7].contiguous())
    keep = torch.ones(capacity, dtype=torch.bool)
    keep[5::7] = False
    _check(hm, keys[keep.to(DEV)])
    hm.erase(keys)
    assert hm.items(return_values=True)[0].shape[0] == 0


@pytest.mark.parametrize("widths", [{"wide": 17}, {"a": 2, "wide": 64}, {f"v{i}": 1 for i in range(5)}])
def test_rows_that_do_not_go_along(ash, widths):
    hm = ash.HashMap(3, widths, 5_000, DEV)
    keys = _keys(0, 3_000)
    hm.insert(keys, {k: torch.rand(3_000, w, device=DEV) for k, w in widths.items()})
    hm.erase(keys[:500])
    _check(hm, keys[500:])


def test_listing_with_a_second_region(ash):
    hm = ash.HashMap(3, {"a": 3, "b": 1}, 5_000, DEV)
    keys = torch.cat([_keys(0, 2_000), _keys(0, 300) + (1 << 24)])
    hm.insert(keys, {"a": torch.rand(2_300, 3, device=DEV), "b": torch.rand(2_300, 1, device=DEV)})
    _check(hm, keys)
    hm.erase(keys[1_900:2_100].contiguous())
    for _ in range(18):
        _check(hm, torch.cat([keys[:1_900], keys[2_100:]]))
    hm.erase(keys[2_100:].contiguous())        # none of them is left
    _check(hm, keys[:1_900])


def test_listings_in_a_graph(ash):
    engine = ash.ASHEngine(3, 8_000, DEV)   # (one workgroup: in order)
    keys = _keys(0, 6_000)
    engine.insert_keys(keys)
    engine.erase(keys[:1_000])
    want = engine.items()
    handle, index = engine.backend._address, engine.backend._index
    host = engine.backend._backend.host
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = host.items(handle, 3, index, 5_000)
    for _ in range(3):
        for t in got:
            t.zero_()
        graph.replay()
        assert all(torch.equal(a, b) for a, b in zip(engine.items(), want))
        assert all(torch.equal(a, b) for a, b in zip(got, want))
