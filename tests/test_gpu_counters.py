"""Counters that an insert or erase leaves for the host itself, in its last
workgroup: against a read of the device (`status`), at the edges of a workgroup and
of the batches that do, with refused keys, tombstones and keys of the second region."""
import warnings

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
LEAVE = 1 << 17   # kLeaveKeys


@pytest.fixture(scope="module")
def ash():
    import ash as module

    return module


def _agree(engine, size):
    """What the host has been told is what the device holds."""
    told = engine.backend.counters()
    assert told["size"] == size
    assert engine.backend.status() == told


def _keys(first, n):
    i = torch.arange(first, first + n, dtype=torch.int32)
    return torch.stack([i % 251, i // 251 % 257, i // (251 * 257)], dim=1).to(DEV)


@pytest.mark.parametrize("n", [1, 255, 256, 257, 1023, 1024, 1025, 70_001, LEAVE, LEAVE + 1])
def test_counters_left_by_inserts_and_erases(ash, n):
    engine = ash.ASHEngine(3, 2 * n + 64, DEV)
    for turn in range(3):   # from the second on, tombstones are looked for
        engine.insert_keys(_keys(0, n))
        _agree(engine, n)
        half = n // 2
        engine.insert_keys(_keys(half, n))   # some stored already
        _agree(engine, n + half)
        engine.erase(_keys(0, n))
        _agree(engine, half)
        engine.erase(_keys(0, n))            # none of them stored
        engine.erase(_keys(n, half) if half else _keys(0, n))
        _agree(engine, 0)


@pytest.mark.parametrize("n", [300, 5_000])
def test_refused_keys_and_tombstones_are_counted(ash, n):
    """A table beyond its capacity: keys are refused, their slots are tombstones."""
    engine = ash.ASHEngine(3, n, DEV)
    for _ in range(2):
        with warnings.catch_warnings(record=True) as seen:
            warnings.simplefilter("always")
            engine.insert_keys(_keys(0, 2 * n))
        assert any(f"{n} keys were not stored" in str(w.message) for w in seen)
        _agree(engine, n)
        assert engine.backend.counters()["tombstones"] > 0
        engine.erase(engine.keys())
        _agree(engine, 0)
        engine.clear()


def test_keys_of_the_second_region_are_counted(ash):
    engine = ash.ASHEngine(3, 4_000, DEV)
    far = _keys(0, 500) + (1 << 24)
    engine.insert_keys(torch.cat([_keys(0, 500), far]))
    _agree(engine, 1_000)
    assert engine.backend.counters()["general_live"] == 500
    engine.erase(far[:200].contiguous())
    _agree(engine, 800)
    assert engine.backend.counters()["general_live"] == 300


def test_erases_in_a_row_and_on_two_streams(ash):
    """Later erases may find the words of an earlier one still owed."""
    engine = ash.ASHEngine(3, 60_000, DEV)
    engine.insert_keys(_keys(0, 50_000))
    side = torch.cuda.Stream()
    for k in range(0, 40_000, 2_000):
        if k % 4_000:
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                engine.erase(_keys(k, 2_000))
            torch.cuda.current_stream().wait_stream(side)
        else:
            engine.erase(_keys(k, 2_000))
    _agree(engine, 10_000)
    left = engine.keys().cpu().numpy()
    want = _keys(40_000, 10_000).cpu().numpy()
    assert np.array_equal(np.unique(left, axis=0), np.unique(want, axis=0))


CHECK = 16 * 256          # keys that a workgroup of the check looks at in its first turns
MOST = 256 * CHECK        # from here on each goes on


@pytest.mark.parametrize("dim, away", [(2, 2**31 - 1), (3, 1 << 20), (4, 1 << 15)])
@pytest.mark.parametrize("n, at", [(1, 0), (256, 255), (CHECK, 17), (CHECK + 1, CHECK), (70_001, 69_999),
                                   (MOST + 300, 5), (MOST + 300, MOST + 299)])
def test_keys_that_do_not_pack_are_met_wherever_they_stand(ash, dim, away, n, at):
    """One key of a batch does not fit the packed code: the insert attaches the second
    region and stores it.  The batch before has none: nothing is attached."""
    # (so much room that no batch streams into a table in use)
    engine = ash.ASHEngine(dim, 12 * n + 64, DEV)
    i = torch.arange(2 * n, dtype=torch.int32, device=DEV)
    keys = torch.zeros(2 * n, dim, dtype=torch.int32, device=DEV)
    edge = {2: 2000, 3: 131, 4: 40}[dim]
    for d in range(dim):
        keys[:, d] = i // edge**d % edge
    engine.insert_keys(keys[:n].contiguous())
    assert engine.backend._general is None
    assert engine.size() == n
    batch = keys[n:].contiguous()
    batch[at] = away
    engine.insert_keys(batch)
    assert engine.backend._general is not None
    _agree(engine, 2 * n)
    assert bool(engine.find(batch)[1].all()) and bool(engine.find(keys[:n].contiguous())[1].all())


def test_inserts_in_a_row_while_others_ask_for_the_size(ash):
    """The words that a call leaves belong to one call at a time: batches that come one
    after the other without a look at the counters, some of them erased again, while
    two threads ask for the size."""
    import threading

    engine = ash.ASHEngine(3, 300_000, DEV)
    for b in range(6):
        engine.insert_keys(_keys(b * 3_001, 3_001))
    _agree(engine, 6 * 3_001)
    over, seen = threading.Event(), []

    def ask():
        with torch.cuda.stream(torch.cuda.Stream()):
            while not over.is_set():
                seen.append(engine.size())

    asking = [threading.Thread(target=ask) for _ in range(2)]
    for t in asking:
        t.start()
    for b in range(40):
        first = 50_000 + b * 1_500
        engine.insert_keys(_keys(first, 1_500))
        if b % 3 == 1:
            engine.erase(_keys(first, 500))
    over.set()
    for t in asking:
        t.join()
    _agree(engine, 6 * 3_001 + 40 * 1_500 - 13 * 500)
    assert all(6 * 3_001 <= n <= 6 * 3_001 + 40 * 1_500 for n in seen)


def test_keys_that_a_full_second_region_refuses_are_reported(ash):
    """A region attached just in case holds 65 536 keys, the table many more."""
    engine = ash.ASHEngine(3, 200_000, DEV)
    engine.insert_keys(_keys(0, 1_000))
    engine.size()
    engine.backend._attach_general(just_in_case=True)
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        engine.insert_keys(_keys(0, 66_000) + (1 << 24))
    assert any("464 keys were not stored" in str(w.message) for w in seen)
    _agree(engine, 66_536)
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        engine.insert_keys(_keys(1_000, 50_000))   # none for the region, which is as full
    assert not seen
    _agree(engine, 116_536)


def test_status_asked_for_beside_an_insert_under_way(ash):
    """A reader of the device on a stream of its own sees the insert that has returned
    before it asks, and what the insert leaves for the host stays there for others.
    (One-dimensional keys: nothing is waited for behind the work in front.)"""
    engine = ash.ASHEngine(1, 20_000, DEV)
    work = torch.randn(8192, 8192, device=DEV)
    keys = torch.arange(16_000, dtype=torch.int32, device=DEV).view(-1, 1)
    one, other = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    for n in (5_000, 16_000):
        with torch.cuda.stream(one):
            for _ in range(8):
                work = torch.tanh(work @ work)
            engine.insert_keys(keys[:n])
        with torch.cuda.stream(other):
            assert engine.backend.status()["size"] == n
            assert engine.size() == n
        assert engine.size() == n
    torch.cuda.synchronize()


def test_readers_beside_calls_that_are_queued_in_parts(ash, monkeypatch):
    """Streaming inserts with keys for the second region and bulk erases, each several
    launches, while others ask for the counters: what those are told in between does not
    stay the latest state, and no key is lost."""
    import threading

    monkeypatch.setattr(ash.common, "BULK_INSERT", "always")
    monkeypatch.setattr(ash.common, "BULK_ERASE", "always")
    engine = ash.ASHEngine(3, 400_000, DEV)
    engine.insert_keys(_keys(0, 70_000))
    over = threading.Event()

    def ask(read):
        with torch.cuda.stream(torch.cuda.Stream()):
            while not over.is_set():
                read()

    asking = [threading.Thread(target=ask, args=(read,)) for read in (engine.size, engine.backend.status)]
    for t in asking:
        t.start()
    try:
        for b in range(12):
            batch = _keys(70_000 + b * 9_000, 70_000)
            batch[::500] += 1 << 24
            engine.insert_keys(batch)
            stored = engine.size()
            assert stored == len(torch.unique(torch.cat([_keys(0, 70_000), batch]), dim=0))
            assert bool(engine.find(batch)[1].all())
            engine.erase(batch)
            assert engine.size() == len(_keys(0, 70_000))
    finally:
        over.set()
        for t in asking:
            t.join()
    _agree(engine, 70_000)


@pytest.mark.parametrize("n", [(3 << 16) - 1, 3 << 16, (3 << 16) + 1, (3 << 16) + 513])
@pytest.mark.parametrize("with_rows", [False, True])
def test_batches_from_which_workgroups_are_larger(ash, n, with_rows):
    """Keys of which a third is stored already, into a table with tombstones and without:
    every key once, under an index of its own, with its own row."""
    m = ash.HashMap(3, {"id": 1}, 10 * n, DEV)
    rows = {"id": torch.arange(n, device=DEV).float().view(-1, 1)}
    stored = _keys(0, n // 3)
    for turn in range(3):
        m.insert(stored, {"id": rows["id"][: n // 3].contiguous()})
        keys = _keys(0, n)
        m.insert(keys, rows) if with_rows else m.engine.insert_keys(keys)
        _agree(m.engine, n)
        idx, masks = m.engine.find(keys)
        assert bool(masks.all()) and len(torch.unique(idx)) == n
        if with_rows:
            assert torch.equal(m.values["id"][idx], rows["id"])
        m.erase(_keys(n // 5, n - n // 5) if turn else keys)
        _agree(m.engine, n // 5 if turn else 0)
        m.erase(_keys(0, n // 5))
