"""Keys looked up, inserted and erased one by one, at the batch sizes where the way a
bucket is read and the size of the workgroups change: what is stored, found and left is
the same on either side, with repeated keys, keys that do not pack, tombstones, and full
buckets on the way."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
STORED = 30_000


@pytest.fixture
def ash(monkeypatch):
    import ash as module
    import ash.common

    monkeypatch.setattr(ash.common, "BULK_INSERT", "never")
    return module


def _keys(n, dim, seed):
    """n distinct keys, a few of them beyond the packed range where there is one."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    i = torch.randperm(n, generator=g, device=DEV) * 11
    if dim == 1:
        return i.int().view(-1, 1).contiguous()
    side = {2: 1 << 12, 3: 1 << 9, 4: 1 << 7}[dim]
    keys = torch.stack([i // side**d % side if d < dim - 1 else i // side**d for d in range(dim)], dim=1).int()
    if dim >= 3:
        keys[i % 997 == 0, 0] += 1 << 28
    return keys.contiguous()


def _rows(n):
    return {"color": torch.rand(n, 3, device=DEV), "id": torch.arange(n, device=DEV).float().view(-1, 1)}


@pytest.mark.parametrize("dim,n", [
    (3, 1), (3, 64), (1, 257), (2, 1025), (4, 5000),
    (1, (5 << 14) - 1), (2, 5 << 14), (3, (5 << 14) + 1), (4, (5 << 14) + 1),
    (3, 5 << 15), (4, (5 << 15) + 1), (1, 3 << 16), (3, (3 << 16) + 1),
    (2, (1 << 18) + 1), (3, (1 << 19) + 3), (3, (3 << 20) + 1)])
def test_batches_come_and_go(ash, dim, n):
    keys = _keys(STORED + n, dim, n)
    stored, new = keys[:STORED].contiguous(), keys[STORED:].contiguous()
    # few buckets to spare, so that many are full
    m = ash.HashMap(dim, {"color": 3, "id": 1}, STORED + n, DEV)
    first = _rows(STORED)
    m.insert(stored, first)
    g = torch.Generator(device=DEV).manual_seed(1)
    twice = torch.randint(n, (n // 10,), generator=g, device=DEV)
    batch = new.clone()
    batch[n - len(twice):] = new[twice]      # repeated keys, others missing
    there = torch.zeros(n, dtype=torch.bool, device=DEV)
    there[: n - len(twice)] = True
    there[twice] = True
    for turn in range(3):   # from the second on among tombstones
        rows = _rows(n)
        m.insert(batch, rows)
        assert m.size() == STORED + int(there.sum())
        masks, found = m.find(new, return_indices=False, return_values=True)
        assert torch.equal(masks, there)
        source = found["id"][:, 0].long()[there]
        assert torch.equal(batch[source], new[there])
        assert torch.equal(found["color"][there], rows["color"][source])
        assert bool((found["color"][~there] == m.values["color"][0]).all())
        # the same from the indices, alone and in a batch that is looked up the other way
        indices, alone = m.engine.find(new)
        many = new.repeat(-(-((1 << 19) + 1) // n), 1) if n <= 1 << 19 else new[: 1 << 18]
        again, masks = m.engine.find(many.contiguous())
        k = min(n, len(many))
        assert torch.equal(alone, there) and torch.equal(masks[:k], there[:k])
        assert torch.equal(again[:k], indices[:k])
        assert torch.equal(m.values["id"][indices[there], 0], found["id"][there, 0])
        both = torch.cat([m.engine.items()[1], m.engine._heap[m.size():].long()])
        assert torch.equal(torch.sort(both)[0], torch.arange(m.engine.capacity, device=DEV))
        m.erase(batch)
        assert m.size() == STORED and not bool(m.engine.find(new)[1].any())
        masks, found = m.find(stored, return_indices=False, return_values=True)
        assert bool(masks.all()) and torch.equal(found["color"], first["color"])
    if n > STORED:   # erased among keys that are not there, the others stay
        m.erase(torch.cat([new[: n - 100], stored[:100]]))
        assert m.size() == STORED - 100 and bool(m.engine.find(stored[100:])[1].all())


@pytest.mark.parametrize("dim,n", [(3, 3 << 14), (2, (3 << 14) + 1), (1, 7 << 14), (4, (7 << 14) + 1), (3, 150_001)])
def test_erases_where_their_workgroups_change(ash, dim, n):
    """The index comes along with the codes of a bucket that other lanes erase from."""
    test_batches_come_and_go(ash, dim, n)


@pytest.mark.parametrize("dim,n", [(3, 5), (1, 1 << 21), (3, 1 << 21), (4, (1 << 21) + 1)])
def test_loads_on_either_side(ash, dim, n):
    """A state dict brought in by lanes alone or by the cooperative probe: every key under
    its index, the others absent."""
    keys = _keys(n + 1000, dim, n)
    engine = ash.HashSet(dim, n + n // 4, DEV).engine
    order = torch.randperm(n, device=DEV)
    state = {"_heap": torch.arange(engine.capacity, dtype=torch.int32, device=DEV),
             "_keys": torch.zeros(engine.capacity, dim, dtype=torch.int32, device=DEV),
             "_indices": torch.zeros(engine.capacity, dtype=torch.int64, device=DEV),
             "_size": torch.tensor([n], dtype=torch.int32, device=DEV)}
    state["_keys"][:n], state["_indices"][:n] = keys[:n], order
    for _ in range(2):   # into a new table, and into one that holds them
        engine.load_state_dict(state)
        assert engine.size() == n
        indices, masks = engine.find(keys)
        assert bool(masks[:n].all()) and not bool(masks[n:].any())
        assert torch.equal(indices[:n], order)
