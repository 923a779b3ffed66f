"""The streaming insert with one split pass: at the edges of its chunks and partitions
and of the batches that split twice, with repeated keys, piles of one key beyond a
partition's capacity, keys that do not pack, batches beyond the capacity, tables that
hold entries or tombstones."""
import warnings

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
CHUNK = 4096
PART = 512 * 6   # capacity of a partition's buckets


@pytest.fixture
def ash(monkeypatch):
    import ash as module
    import ash.common

    monkeypatch.setattr(ash.common, "BULK_INSERT", "always")
    return module


def _keys(first, n, dim=3):
    i = torch.arange(first, first + n, dtype=torch.int64, device=DEV)
    i = (i * 2654435761) % (1 << 30)          # (distinct: the factor is odd)
    if dim == 1:
        return i.int().view(-1, 1).contiguous()
    if dim == 2:
        return torch.stack([i % 40_000, i // 40_000], dim=1).int().contiguous()
    if dim == 3:
        return torch.stack([i % 1024, i // 1024 % 1024, i // (1 << 20)], dim=1).int().contiguous()
    return torch.stack([i % 128, i // 128 % 128, i // (1 << 14) % 256, i // (1 << 22)], dim=1).int().contiguous()


def _check(m, distinct, values=None, capacity=None):
    """Every distinct key is stored once, indices in use and the free list are every
    index once, and a key's rows are those of one of its rows in the batch."""
    n = distinct.shape[0]
    assert m.size() == n == m.engine.backend.status()["size"]
    idx, masks = m.engine.find(distinct)
    assert bool(masks.all())
    both = torch.cat([m.engine.items()[1], m.engine._heap[n:].long()])
    assert torch.equal(torch.sort(both)[0], torch.arange(m.engine.capacity, device=DEV))
    assert torch.equal(torch.sort(idx)[0], torch.sort(m.engine.items()[1])[0])
    if values is not None:
        keys, rows = values
        source = m.values["id"][idx, 0].long()
        assert torch.equal(keys[source], distinct)
        assert torch.equal(m.values["color"][idx], rows["color"][source])


def _rows(n):
    return {"color": torch.rand(n, 3, device=DEV), "id": torch.arange(n, device=DEV).float().view(-1, 1)}


@pytest.mark.parametrize("dim", [1, 2, 3, 4])
@pytest.mark.parametrize("n", [CHUNK, CHUNK + 1, 3 * CHUNK - 1, 50_001])
@pytest.mark.parametrize("with_rows", [False, True])
def test_new_tables(ash, dim, n, with_rows):
    distinct = _keys(0, n, dim)
    perm = torch.randperm(n + n // 2, device=DEV)
    keys = torch.cat([distinct, distinct[: n // 2]])[perm].contiguous()
    if with_rows:
        m, rows = ash.HashMap(dim, {"color": 3, "id": 1}, 2 * n, DEV), _rows(len(keys))
        m.insert(keys, rows)
        _check(m, distinct, (keys, rows))
    else:
        m = ash.HashSet(dim, 2 * n, DEV)
        m.insert(keys)
        _check(m, distinct)


@pytest.mark.parametrize("capacity", [100, PART, PART + 1, 8 * PART, 8 * PART + 1, 9 * PART])
def test_few_partitions(ash, capacity):
    """Tables of one partition, of a short one, of as many as XCDs and one more."""
    n = capacity - capacity // 8
    distinct = _keys(0, n)
    keys = distinct[torch.arange(max(n, CHUNK) + 77, device=DEV) % n].contiguous()
    m = ash.HashMap(3, {"color": 3, "id": 1}, capacity, DEV)
    rows = _rows(len(keys))
    m.insert(keys, rows)
    _check(m, distinct, (keys, rows))


@pytest.mark.parametrize("n, capacity", [
    (1024 * CHUNK, 6_000_000),            # the most chunks
    (1024 * CHUNK + 1, 6_000_000),        # split twice
    (300_000, 4096 * PART),               # the most partitions
    (300_000, 4096 * PART + 1),           # split twice
])
def test_bounds_of_one_pass(ash, n, capacity):
    keys = _keys(0, n)
    m = ash.HashMap(3, {"color": 3, "id": 1}, capacity, DEV)
    rows = _rows(n)
    m.insert(keys, rows)
    _check(m, keys, (keys, rows))
    s = ash.HashSet(3, capacity, DEV)
    s.insert(keys)
    assert s.size() == n and bool(s.find(keys).all())


@pytest.mark.parametrize("with_rows", [False, True])
@pytest.mark.parametrize("erased", [0, 9_000])
def test_tables_that_hold_entries(ash, with_rows, erased):
    """Entries and, once keys are gone, a heap out of order and tombstones."""
    old, new = _keys(0, 40_000), _keys(30_000, 40_000)
    if with_rows:
        m = ash.HashMap(3, {"color": 3, "id": 1}, 71_000, DEV)
        m.insert(old, {"color": torch.zeros(40_000, 3, device=DEV), "id": torch.full((40_000, 1), -1.0, device=DEV)})
    else:
        m = ash.HashSet(3, 71_000, DEV)
        m.insert(old)
    if erased:
        m.erase(old[:erased])
    for _ in range(2):
        if with_rows:
            rows = _rows(40_000)
            m.insert(new, rows)
        else:
            m.insert(new)
    distinct = _keys(erased, 70_000 - erased)
    _check(m, distinct)
    if with_rows:
        idx, _ = m.engine.find(new)
        ids = m.values["id"][idx, 0]
        assert bool((ids[:10_000] == -1).all())       # stored already: rows left alone
        assert torch.equal(ids[10_000:], torch.arange(10_000, 40_000, device=DEV).float())


@pytest.mark.parametrize("with_rows", [False, True])
def test_piles_of_one_key(ash, with_rows):
    """More copies of a key than a partition's records have room."""
    distinct = _keys(0, 20_000)
    keys = torch.cat([distinct, distinct[:1].expand(30_000, 3), distinct[7:8].expand(5_000, 3)])
    keys = keys[torch.randperm(len(keys), device=DEV)].contiguous()
    if with_rows:
        m, rows = ash.HashMap(3, {"color": 3, "id": 1}, 60_000, DEV), _rows(len(keys))
        m.insert(keys, rows)
        _check(m, distinct, (keys, rows))
    else:
        m = ash.HashSet(3, 60_000, DEV)
        m.insert(keys)
        _check(m, distinct)


@pytest.mark.parametrize("with_rows", [False, True])
@pytest.mark.parametrize("ranges", [512, 513, 1300])
@pytest.mark.parametrize("per_bucket, copies", [(0.5, 1), (3, 2), (4.5, 1), (4.5, 40), (3, 4000)])
def test_ranges_built_from_lists(ash, with_rows, ranges, per_bucket, copies):
    """Emptied tables on both sides of the number of ranges and of the records per
    bucket from which ranges are built from lists: buckets that overflow, keys that
    repeat beyond a bucket's slots, beyond what is placed beside the list, beyond a
    range's records."""
    capacity, n = ranges * PART, int(ranges * 512 * per_bucket)
    distinct = _keys(7, max(n // copies, n - 40_000) if copies == 4000 else n // copies)
    if copies == 4000:   # piles of a few keys among many
        keys = torch.cat([distinct, distinct[:10].repeat(4000, 1)[: n - len(distinct)]])
    else:
        keys = distinct.repeat(copies, 1)
    keys = keys[torch.randperm(len(keys), device=DEV)].contiguous()
    if with_rows:
        m, rows = ash.HashMap(3, {"color": 3, "id": 1}, capacity, DEV), _rows(len(keys))
        m.insert(keys, rows)
        _check(m, distinct, (keys, rows))
    else:
        m = ash.HashSet(3, capacity, DEV)
        m.insert(keys)
        _check(m, distinct)
    absent = _keys(100_000_000, 50_000)
    assert not bool(m.engine.find(absent)[1].any())
    m.engine.erase(distinct[::2].contiguous())
    _check(m, distinct[1::2].contiguous())


@pytest.mark.parametrize("with_rows", [False, True])
def test_keys_that_do_not_pack_and_batches_beyond_the_capacity(ash, with_rows):
    far = _keys(0, 700) + (1 << 24)
    distinct = torch.cat([_keys(0, 9_000), far])
    keys = distinct[torch.randperm(len(distinct), device=DEV)].contiguous()
    make = (lambda c: ash.HashMap(3, {"color": 3, "id": 1}, c, DEV)) if with_rows else (lambda c: ash.HashSet(3, c, DEV))
    m, rows = make(12_000), _rows(len(keys))
    m.insert(keys, rows) if with_rows else m.insert(keys)
    assert m.size() == len(distinct) and bool(m.engine.find(distinct)[1].all())
    if with_rows:
        idx, _ = m.engine.find(keys)
        assert torch.equal(m.values["color"][idx], rows["color"])
    small = make(5_000)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        small.insert(_keys(0, 9_000), _rows(9_000)) if with_rows else small.insert(_keys(0, 9_000))
    assert small.size() == 5_000
    assert int(small.engine.find(_keys(0, 9_000))[1].sum()) == 5_000


def test_replays_of_a_streamed_insert(ash):
    """Captured: the launch's place among the counters is zero after every replay."""
    s = ash.HashSet(3, 40_000, DEV)
    keys = _keys(0, 20_000)
    s.insert(keys)
    s.erase(keys)
    host, handle, index = s.engine.backend._backend.host, s.engine.backend._address, s.engine.backend._index
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        host.insert(handle, 3, index, 40_000, keys, [], [], [], 1)
    for _ in range(4):
        graph.replay()
        assert s.size() == 20_000 and bool(s.find(keys).all())
        s.erase(keys[:5_000])
        s.insert(_keys(20_000, 8_000))
        s.erase(_keys(5_000, 23_000))
        assert s.size() == 0


def test_which_batches_stream():
    """The bars of ASH_STREAMING_EARLY (3) on new tables and on tables in use, and what
    ASH_STREAMING_AUTO (0) says to the same: scratch is asked for or not.  Smaller
    batches, those with rows and those into tables in use lose where keys repeat or are
    stored already."""
    import ctypes

    import ash

    def wanted(engine, n, rows=()):
        """(under ASH_STREAMING_EARLY, under ASH_STREAMING_AUTO)"""
        nbytes = ctypes.c_int64(-1)
        widths = (ctypes.c_int64 * max(1, len(rows)))(*rows)
        backend, both = engine.backend, []
        for policy in (3, 0):
            backend._check(backend._lib.ash_map_insert_scratch_bytes(
                backend._handle, n, len(rows), widths if rows else None, policy, ctypes.byref(nbytes)))
            both.append(nbytes.value > 0)
        return tuple(both)

    yes, no, early = (True, True), (False, False), (True, False)
    engine = ash.ASHEngine(3, 300_000, DEV)          # 50 176 buckets
    assert wanted(engine, 1 << 17) == early and wanted(engine, (1 << 17) - 1) == no
    assert wanted(engine, (1 << 18) - 1) == early and wanted(engine, 1 << 18) == yes
    assert wanted(engine, (1 << 18) - 1, (12, 4)) == no and wanted(engine, 1 << 18, (12, 4)) == yes
    assert wanted(engine, 13 * 50_176) == no         # piles
    wide = ash.ASHEngine(3, 1_200_000, DEV)          # 200 192 buckets
    assert wanted(wide, 200_191) == no and wanted(wide, 200_192) == early
    large = ash.ASHEngine(3, 4_000_000, DEV)         # 667 136 buckets
    assert wanted(large, 1 << 18) == yes
    assert wanted(large, 1 << 18, (12, 4)) == no and wanted(large, 340_000, (12, 4)) == yes
    for each in (engine, wide, large):
        each.find(_keys(0, 10))                      # in use from here on
        assert wanted(each, 1 << 18) == no and wanted(each, 400_000, (12, 4)) == no
    assert wanted(large, 660_000) == no and wanted(large, 1 << 20) == yes
