"""What the host keeps of a map's counters while calls and readers meet, one
function a test of test_host_counters.py (each in a process of its own)."""
import time

from stand_in_device import (ALWAYS, DROPPED, EXOTIC, SIZE, Map, beside)

ONE, OTHER = 0x10, 0x20   # streams


def _queued_insert(device):
    """A map with an insert of 100 keys that is still under way on stream ONE."""
    m = Map(device, key_dim=1)   # (nothing to wait for in one dimension)
    device.stream(ONE).hold()
    device.effects = [{SIZE: 100}]
    assert m.insert(stream=ONE) == 0 and m.pending()
    return m


def status_beside_an_insert_under_way(device):
    """A reader that asks the device has the words of the insert that is under way
    before it, and leaves them to the others."""
    m = _queued_insert(device)
    asked = beside(lambda: m.status(OTHER))
    time.sleep(0.1)
    device.stream(ONE).go()
    asked.join()
    assert (asked.result, m.size(OTHER), m.size(ONE)) == (100, 100, 100)
