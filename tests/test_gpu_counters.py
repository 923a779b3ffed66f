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
