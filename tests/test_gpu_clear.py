"""HashMap.clear in one launch: counters, heap, log, the bucket array of small tables and
the value rows, over odd sizes, types, numbers of values and states of the map."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
# tables of up to 42 probe ranges are filled by the clear itself (kFillAtOnce)
EDGE = 42 * 512 * 6


@pytest.fixture(scope="module")
def ash():
    import ash as module

    return module


def _keys(first, n):
    i = torch.arange(first, first + n, dtype=torch.int32)
    return torch.stack([i % 251, i // 251 % 257, i // (251 * 257)], dim=1).to(DEV)


@pytest.mark.parametrize("capacity", [1, 3, 64, 1365, 1366, 50_001, EDGE, EDGE + 1])
@pytest.mark.parametrize("erased", [False, True])
def test_clear_empties_the_map_and_zeroes_its_rows(ash, capacity, erased):
    widths = {"a": 1, "b": 3, "c": 7, "d": 2, "e": 5}   # the fifth is beyond one launch's
    hm = ash.HashMap(3, widths, capacity, DEV)
    n = capacity
    for turn in range(2):
        rows = {k: torch.rand(n, w, device=DEV) + 1 for k, w in widths.items()}
        hm.insert(_keys(turn, n), rows)
        assert hm.size() == n
        if erased:
            hm.erase(_keys(turn, max(1, n // 3)))
        versions = {k: v._version for k, v in hm.values.items()}
        hm.clear()
        assert all(v._version > versions[k] for k, v in hm.values.items())
        assert hm.size() == 0 and hm.keys().shape[0] == 0
        for rows in hm.values.values():
            assert not bool(rows.any())
        masks, _ = hm.engine.find(_keys(0, n + 1))[::-1]
        assert not bool(masks.any())
        assert torch.equal(torch.sort(hm.engine._heap)[0].cpu(), torch.arange(capacity, dtype=torch.int32))
    hm.insert(_keys(5, n), {k: torch.ones(n, w, device=DEV) for k, w in widths.items()})
    assert hm.engine.backend.status()["size"] == n
    assert torch.equal(torch.sort(hm.items()[1])[0].cpu(), torch.arange(n))


def test_rows_that_torch_has_to_zero(ash):
    """Types of one byte and rows of odd sizes go along; a tensor that is strided,
    misaligned or takes part in autograd is zeroed by torch, or refused by it."""
    hm = ash.HashMap(2, {"a": 1, "b": 2, "c": 4, "d": 1}, 1001, DEV)
    flags = torch.ones(1001, 1, dtype=torch.bool, device=DEV)
    strided = torch.ones(1001, 4, device=DEV)[:, ::2]
    shifted = torch.ones(4 * 1001 + 1, device=DEV)[1:].view(1001, 4)
    guard = torch.ones(1001 + 7, dtype=torch.uint8, device=DEV)
    hm.values.update(a=flags, b=strided, c=shifted, d=guard[:1001].view(-1, 1))
    hm.clear()
    assert not any(bool(t.any()) for t in hm.values.values())
    assert bool(guard[1001:].all())          # nothing behind the rows
    leaf = torch.ones(1001, 1, device=DEV, requires_grad=True)
    hm.values["a"] = leaf
    with pytest.raises(RuntimeError):
        hm.clear()
    with torch.no_grad():
        hm.clear()
    assert not bool(leaf.any())


@pytest.mark.parametrize("capacity", [3_000, EDGE + 600])
def test_clear_in_a_graph(ash, capacity):
    """Replays empty the map whatever was inserted in between."""
    hm = ash.HashMap(3, 4, capacity, DEV)
    keys, rows = _keys(0, 2_000), torch.rand(2_000, 4, device=DEV)
    hm.insert(keys, rows)
    hm.find(keys)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        hm.clear()
    for turn in range(4):
        hm.insert(keys, rows)
        assert hm.size() == 2_000
        if turn % 2:
            hm.erase(keys[:700])
        graph.replay()
        torch.cuda.synchronize()
        assert hm.size() == 0 and not bool(hm.values["default"].any())
        assert not bool(hm.find(keys)[0].any())
