"""What the host keeps of a map's counters while calls and readers meet, one
function a test of test_host_counters.py (each in a process of its own)."""
import re
import time

from stand_in_device import ALWAYS, DROPPED, EXOTIC, I64, INT, LIBRARY, PTR, SIZE, TOMBS, Map, beside

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


def _stands_at(m, size):
    """The size as the handle keeps it, on either stream, and as the device has it."""
    seen = m.size(ONE), m.size(OTHER), m.status(ONE)
    assert seen == (size,) * 3, seen


def a_reader_on_another_stream_than_the_change(device):
    """What a stream sees that does not wait for the change is not kept."""
    m = Map(device)
    device.stream(ONE).hold()
    device.effects = [{SIZE: 7}]
    assert m.activate(ONE) == 0
    assert m.size(OTHER) == 0
    device.stream(ONE).go()
    _stands_at(m, 7)


def _read_before(device, m, kernel):
    """A reader that has its answer just before `kernel` is queued on its stream."""

    def read():
        reader = beside(lambda: m.size(ONE))
        reader.join()
        assert reader.result is not None

    device.before[kernel] = read


def a_reader_before_the_launch_of_an_activation(device):
    m = Map(device)
    device.effects = [{SIZE: 7}]
    _read_before(device, m, "activate_runs_kernel")
    assert m.activate(ONE) == 0
    _stands_at(m, 7)


def a_reader_before_the_launch_of_a_bulk_erase(device):
    m = Map(device)
    device.effects = [{SIZE: 700}, {SIZE: -600}]
    assert m.activate(ONE) == 0
    _read_before(device, m, "erase_range_kernel")
    assert m.erase_bulk(stream=ONE) == 0
    _stands_at(m, 100)


def a_reader_before_the_last_launches_of_a_streaming_insert(device):
    """Keys that wait for the second region are reported, whatever a reader was told
    while the insert was being queued."""
    m = Map(device)
    device.spilled = 5
    device.effects = [{SIZE: 70_000, EXOTIC: 5}]
    _read_before(device, m, "build_kernel")
    assert m.insert(70_000, ALWAYS, ONE) == 2   # ASH_NEEDS_GENERAL
    assert device.ctr[SIZE] == 70_000
    _stands_at(m, 70_000)


def _answer_across(device, m, call):
    """A reader whose answer is from before `call` and comes after it has returned."""
    device.stream(OTHER).hold()
    reader = beside(lambda: m.size(OTHER))
    while not device.stream(OTHER).queue:
        time.sleep(0.001)
    device.stream(ONE).hold()
    assert call() == 0
    device.stream(OTHER).go()
    reader.join()
    device.stream(ONE).go()
    return reader.result


def a_reader_across_a_clear(device):
    m = Map(device)
    device.effects = [{SIZE: 7}]
    assert m.activate(OTHER) == 0
    assert _answer_across(device, m, lambda: m.clear(ONE)) == 7
    _stands_at(m, 0)


def a_reader_across_a_load(device):
    m = Map(device)
    device.effects = [{SIZE: 7}]
    assert m.activate(OTHER) == 0
    assert _answer_across(device, m, lambda: m.load(3, ONE)) == 7
    _stands_at(m, 3)


def a_reader_across_a_rebuild(device):
    """(the tombstones go: the status has them)"""
    m = Map(device)
    device.effects = [{SIZE: 7, TOMBS: 5}]
    assert m.activate(OTHER) == 0
    assert _answer_across(device, m, lambda: m.rebuild(ONE)) == 7
    assert m.counters(ONE)[2] == 0


def words_under_way_when_the_second_region_comes(device):
    """The size is that of the insert before, wherever it is asked for."""
    m = _queued_insert(device)
    attached = beside(lambda: m.attach(ONE))
    time.sleep(0.1)
    seen = beside(lambda: m.size(OTHER))
    time.sleep(0.1)
    device.stream(ONE).go()
    attached.join(), seen.join()
    assert (attached.result, seen.result) == (0, 100)
    _stands_at(m, 100)


def keys_that_the_second_region_refuses(device):
    """A batch with keys for the second region: the region may be full while the table
    is not, so the counters have been read when the insert returns."""
    m = Map(device)
    assert m.attach() == 0
    device.bad_keys, device.effects = 3, [{SIZE: 80, DROPPED: 20}]
    assert m.insert() == 0 and not m.pending()
    assert m.counters()[:2] == [80, 20]
    device.bad_keys, device.effects = 0, [{SIZE: 100}]
    assert m.insert() == 0 and m.pending()
    assert m.counters()[:2] == [180, 20]


def _lines(device, stream):
    return {word // 128 for on, word in device.words if on == stream}


def a_streaming_insert_that_fails_behind_its_first_launch(device):
    """(the word of its first pass is owed)"""
    m = Map(device)
    device.stream(ONE).hold()
    device.refuse = ("build_kernel",)
    assert m.insert(70_000, ALWAYS, ONE) == 1
    device.refuse = ()
    device.effects = [{SIZE: 70_000}]
    assert m.insert(70_000, ALWAYS, OTHER) == 0
    assert not _lines(device, ONE) & _lines(device, OTHER)
    device.stream(ONE).go()
    assert m.size(OTHER) == 70_000


def a_map_that_goes_with_words_owed(device):
    """The line of a failed call serves no other map."""
    m = Map(device, key_dim=1)
    device.stream(ONE).hold()
    device.refuse = ("scatter_rows_kernel",)
    assert m.insert(stream=ONE, values=1, row_bytes=4096) == 1
    device.refuse = ()
    assert m.lib.ash_map_destroy(m.handle) == 0
    others = [Map(device, key_dim=1) for _ in range(3)]
    for other in others:
        assert other.insert(stream=OTHER) == 0
    assert not _lines(device, ONE) & _lines(device, OTHER)
    device.stream(ONE).go()


def inserts_that_are_refused_before_their_launch(device):
    """They owe nothing: their lines serve the next call."""
    m = Map(device)
    for _ in range(3):
        assert m.insert() == 0
    used = _lines(device, 0)
    for _ in range(100):
        assert m.insert(values=1, row_bytes=0) == 1   # (no value rows)
        assert m.insert() == 0
    assert _lines(device, 0) == used


def a_frame_whose_count_fails(device):
    """It is integrated all the same: its flags, left up, would have the next frame
    integrate and count its blocks as well."""
    m = Map(device)
    device.refuse = ("count_flags_kernel",)
    assert m.fuse() == 1
    assert any("integrate_depth_flagged_kernel" in name for name in device.launched)
    device.refuse = ()
    assert m.fuse() == 0


def scratch_of_rays_that_are_captured_is_not_kept(device):
    """Whether the call's own stream is captured: not that of the device which is current."""
    m = Map(device)
    kept = m.lib.ash_ray_volume_kept
    ask = lambda stream: kept(m.handle, PTR(stream))
    assert [ask(s) for s in (0, ONE, OTHER)] == [1, 1, 1] and kept(PTR(0), PTR(ONE)) == 0
    for current in (0, 1):
        for captured in (0, ONE):
            device.runtime.stand_in_capture(2, current, 0, PTR(captured))
            assert [ask(s) for s in (0, ONE, OTHER)] == [int(s != captured) for s in (0, ONE, OTHER)]
            assert device.runtime.stand_in_current_device() == current
            # (a capture of the other device's default stream is none of this map's)
            device.runtime.stand_in_capture(2, current, 1, PTR(0))
            assert ask(0) == 1


def as_many_rays_as_gain_their_volume_back(device):
    """More where the call clears it than where it is kept, and beside a long log."""
    short, long = Map(device, capacity=100_000), Map(device, capacity=3_000_000)
    cleared, kept = device.lib.ash_ray_volume_bytes, device.lib.ash_map_ray_volume_bytes
    cleared.restype = kept.restype = I64
    has = lambda n, sampling, hi=31: cleared(INT(0), INT(hi), I64(n), INT(sampling)) > 0
    keeps = lambda m, n, samples, hi=31: kept(m.handle, INT(0), INT(hi), I64(n), I64(samples)) > 0
    assert [has(n, 0) for n in (0, 1024, 4095, 4096)] == [False, False, False, True]
    assert [has(n, 1) for n in (0, 2048, 8191, 8192)] == [False, False, False, True]
    assert [keeps(short, n, 0) for n in (1023, 1024, 4095, 4096)] == [False, True, True, True]
    assert [keeps(long, n, 0) for n in (1024, 4095, 4096)] == [False, False, True]
    for samples in (1, 16, 63):
        assert [keeps(m, n, samples) for m in (short, long) for n in (8191, 8192)] == [False, True] * 2
    for samples in (64, 128, 1 << 40):
        assert [keeps(short, n, samples) for n in (2047, 2048, 8191, 8192)] == [False, True, True, True]
        assert [keeps(long, n, samples) for n in (2048, 7812, 7813, 8192)] == [False, False, True, True]
    assert not has(1 << 20, 0, 161) and not keeps(short, 1 << 20, 0, 161) and not keeps(short, 1 << 20, 0, -1)


def larger_workgroups_only_where_they_are_launched(device):
    """Inserts of keys, with rows and without (modes 0 and 1)."""
    wide = {name.split("insert_kernelI")[1][:10] for name in device.kernels()
            if "insert_kernelI" in name and "Li512E" in name}
    assert wide == {f"Li{dim}ELi{mode}ELb" for dim in (1, 2, 3, 4) for mode in (0, 1)}, wide


def every_kernel_that_is_built_is_launched_from_somewhere(device):
    """(the device code holds what a template names, also where its launch is never compiled)"""
    with open(LIBRARY, "rb") as f:
        built = {name.decode() for name in re.findall(rb"(_Z\w+)\.kd\0", f.read())}
    registered = set(device.kernels())
    assert len(built) > 100 and built == registered, built ^ registered


def backward_kernels_only_of_widths_that_are_launched(device):
    """A lane per channel, eight lanes a query: rows of five to eight, which go by rows in
    single precision."""
    by_channel = [name for name in device.kernels() if "query_backward_" in name and "_vec_kernel" not in name]
    assert any("IdLi8E" in name for name in by_channel) and any("IfLi16E" in name for name in by_channel)
    assert not [name for name in by_channel if "IfLi8E" in name]
    # eight wavefronts to a table of cells: rows of up to eight that are scattered
    wide = {int(name.split("_vec_kernelILi")[1].split("E")[0]) for name in device.kernels()
            if "_vec_kernelI" in name and "Li512E" in name}
    assert wide == set(range(1, 9)), wide
    # gradients of queries alone: all widths but that of one channel
    alone = {int(name.split("_vec_kernelILi")[1].split("E")[0]) for name in device.kernels()
             if re.search(r"_vec_kernelILi\d+ELb[01]ELi2E", name)}
    assert alone == {2, 3, 4, 5, 6, 7, 8, 12, 16}, alone


def programs_that_interpolate_do_not_load_the_backward_by_rows(device):
    """The runtime loads a device code with the first of its kernels: every width's by
    rows has one of its own."""
    with open(LIBRARY, "rb") as f:
        codes = f.read().split(b"\x7fELF")[2:]   # (the library itself comes first)
    kernels = [{name.decode() for name in re.findall(rb"(_Z\w+)\.kd\0", code)} for code in codes]
    by_rows = [names for names in kernels if any("_vec_kernelI" in name for name in names)]
    widths = [{name.split("_vec_kernelILi")[1].split("E")[0] for name in names} for names in by_rows]
    assert sorted(int(width) for width, in widths) == [1, 2, 3, 4, 5, 6, 7, 8, 12, 16], widths
    assert any("grid_forward_kernel" in name for names in kernels for name in names)
