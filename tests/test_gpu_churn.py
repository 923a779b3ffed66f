"""Keys that come and go next to a full stretch of the table: the slots they
leave behind are taken again, so that the stretch does not grow until its probe
range is full and keys are refused although the map has room."""
import pytest
import torch

import ash.common as common

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
CAPACITY = 20_000
BUCKETS, RANGE = 3584, 512     # of such a map, and of a probe range
M64 = (1 << 64) - 1


def _home(x, y, z):
    """The bucket a key's sequence starts at."""
    h = (x + (1 << 20)) | ((y + (1 << 20)) << 21) | ((z + (1 << 20)) << 42)
    h ^= h >> 33
    h = h * 0xFF51AFD7ED558CCD & M64
    h ^= h >> 33
    h = h * 0xC4CEB9FE1A85EC53 & M64
    h ^= h >> 33
    return ((h >> 32) * BUCKETS) >> 32


def _keys_near(first, width, n, ranges=1):
    """n keys per range whose home buckets lie in first .. first + width - 1."""
    found = [[] for _ in range(ranges)]
    i = 0
    while min(len(f) for f in found) < n:
        key = (i % 1000, i // 1000, 7)
        i += 1
        r, at = divmod(_home(*key), RANGE)
        if r < ranges and first <= at < first + width and len(found[r]) < n:
            found[r].append(key)
    return torch.tensor([f for part in zip(*found) for f in part], dtype=torch.int32, device=DEV)


def _tombstones(gpu_ash, engine):
    return gpu_ash.core.backend.host.counters(engine.backend._address, engine.backend._index)[2]


# one stretch and the per-key kernel; one per range, by the streaming insert
@pytest.mark.parametrize("policy,width,stored,coming,ranges", [
    ("never", 10, 85, 60, 1), ("never", 1, 9, 5000 // RANGE, 1), ("always", 60, 510, 600, 7)])
def test_keys_that_come_and_go(gpu_ash, monkeypatch, policy, width, stored, coming, ranges):
    monkeypatch.setattr(common, "BULK_INSERT", policy)
    near = _keys_near(100, width, stored + coming, ranges)
    engine = gpu_ash.ASHEngine(3, CAPACITY, DEV)
    engine.insert_keys(near[:stored * ranges])
    come = near[stored * ranges:]
    g = torch.Generator(device=DEV).manual_seed(1)
    left = []
    for _ in range(100):
        engine.insert_keys(come[torch.randperm(len(come), generator=g, device=DEV)])
        assert engine.size() == len(near)
        engine.erase(come[torch.randperm(len(come), generator=g, device=DEV)])
        left.append(_tombstones(gpu_ash, engine))
    indices, masks = engine.find(near)
    assert engine.size() == stored * ranges and int(masks.sum()) == stored * ranges
    assert bool(masks[:stored * ranges].all())
    assert len(torch.unique(indices[masks])) == stored * ranges
    # no more than one batch leaves, whatever its order (at first: none stood there)
    assert max(left) <= len(come) and left[-1] <= left[0] + 10 * ranges, left


@pytest.mark.parametrize("policy", ["never", "always"])
def test_copies_of_a_key_meet_in_one_freed_slot(gpu_ash, monkeypatch, policy):
    """Each key eight times in a batch that goes to a stretch of tombstones."""
    monkeypatch.setattr(common, "BULK_INSERT", policy)
    near = _keys_near(100, 60, 1000, 7)
    engine = gpu_ash.ASHEngine(3, CAPACITY, DEV)
    g = torch.Generator(device=DEV).manual_seed(2)
    for _ in range(6):
        engine.insert_keys(near)
        gone = near[torch.randperm(len(near), generator=g, device=DEV)[:3500]]
        engine.erase(gone)
        assert _tombstones(gpu_ash, engine) > 0
        again = gone.repeat(8, 1)
        engine.insert_keys(again[torch.randperm(len(again), generator=g, device=DEV)])
        assert engine.size() == len(near)
        keys, indices = engine.items()
        assert len(torch.unique(keys, dim=0)) == len(torch.unique(indices)) == len(near)
        indices, masks = engine.find(near)
        assert bool(masks.all()) and len(torch.unique(indices)) == len(near)


@pytest.mark.parametrize("n", [1, 9, 10, 11, 21])
def test_copies_of_the_keys_of_one_bucket(gpu_ash, monkeypatch, n):
    """A bucket's ten slots, tried by every key from one of its own on: keys of one home
    bucket, each a hundred times in the batch, into an empty map, beside half of them,
    and behind what was erased."""
    monkeypatch.setattr(common, "BULK_INSERT", "never")
    near = _keys_near(100, 1, n)
    engine = gpu_ash.ASHEngine(3, CAPACITY, DEV)
    g = torch.Generator(device=DEV).manual_seed(n)
    for gone in (n, (n + 1) // 2, 1):
        batch = near.repeat(100, 1)
        engine.insert_keys(batch[torch.randperm(len(batch), generator=g, device=DEV)])
        keys, indices = engine.items()
        assert engine.size() == n == len(torch.unique(keys, dim=0)) == len(torch.unique(indices))
        found, masks = engine.find(near)
        filed = torch.zeros(CAPACITY, 3, dtype=torch.int32, device=DEV)
        filed[indices] = keys
        assert bool(masks.all()) and torch.equal(filed[found], near)
        engine.erase(near[:gone])
        assert engine.size() == n - gone


def test_refused_keys_leave_slots_that_later_inserts_take(gpu_ash, monkeypatch):
    """Inserts that do not look for tombstones (none known), into a full map whose
    refused keys have left some, with copies; then those that do, captured ones
    and replays among them."""
    monkeypatch.setattr(common, "BULK_INSERT", "never")
    near = _keys_near(100, 40, 380, 1)
    engine = gpu_ash.ASHEngine(3, 330, DEV)

    def stored():
        keys, indices = engine.items()
        assert len(torch.unique(keys, dim=0)) == len(torch.unique(indices)) == engine.size()
        found, masks = engine.find(near)
        assert int(masks.sum()) == engine.size() == len(torch.unique(found[masks]))
        return engine.size()

    for _ in range(3):                       # 50 keys are refused each time
        engine.insert_keys(near.repeat(4, 1))
        assert stored() == 330
    for turn in range(4):
        engine.erase(near[turn * 20:turn * 20 + 200])
        engine.insert_keys(near[turn * 20 + 30:turn * 20 + 130].repeat(3, 1))
        assert stored() <= 330
    engine.erase(near)
    assert stored() == 0
    engine.insert_keys(near[:300])
    assert stored() == 300
    few = near[250:300].repeat(2, 1)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    engine.erase(few)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        engine.backend.insert_keys(few)       # (everything is loaded before the capture)
        engine.erase(few)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            engine.backend.insert_keys(few)
    torch.cuda.synchronize()
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert stored() == 300
        engine.erase(few)
        assert stored() == 250
