"""libash_hip.so on a CPU, its launches done by this file: for tests of what the
host side keeps of the counters.

    python tests/stand_in_device.py STAND_IN_LIBRARY SCENARIO

runs one of host_scenarios.py (test_host_counters.py) in a process without torch, so
that the stand-in's entry points are found before the HIP runtime's.
"""
import ctypes
import os
import struct
import sys
import threading
import time

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBRARY = os.path.join(ROOT, "torch-ash_amd", "ash", "lib", "libash_hip.so")
# the counters as the table's header has them
SIZE, TOMBS, DROPPED, EXOTIC, GEN_LIVE, TOUCHED = 0, 1, 2, 3, 5, 6
HOST_COUNTERS = 8
AUTO, ALWAYS, NEVER, EARLY = range(4)
PTR, I32, I64, INT = ctypes.c_void_p, ctypes.c_int32, ctypes.c_int64, ctypes.c_int


def _i32(value):
    return struct.unpack("<i", struct.pack("<I", value & 0xFFFFFFFF))[0]


def _words(address):
    return (ctypes.c_uint64 * HOST_COUNTERS).from_address(address)


class Stream:
    """Work is done where it is queued, or, while the stream is held, on `go`."""

    def __init__(self):
        self.held, self.queue = False, []

    def hold(self):
        self.held = True

    def go(self):
        self.held = False
        while self.queue:
            self.queue.pop(0)()


class Device:
    def __init__(self, stand_in):
        self.runtime = ctypes.CDLL(stand_in, mode=ctypes.RTLD_GLOBAL)
        self.streams = {}
        self.launched = []        # names
        self.words = []           # (stream, address) of words that launches are to leave
        self.refuse = ()          # parts of the names of kernels whose launch fails
        self.before = {}          # part of a kernel's name -> called (once) where it is launched
        self.no_host_memory = False
        # what inserts, erases and activations do to the counters
        self.effects = []
        self.bad_keys = 0         # keys that do not fit the packed code
        self.spilled = 0          # keys that a streaming insert hands to the per-key kernel
        self._callbacks = (ctypes.CFUNCTYPE(INT, ctypes.c_char_p, ctypes.c_size_t, ctypes.POINTER(PTR))(self._launch),
                           ctypes.CFUNCTYPE(INT, ctypes.c_size_t)(self._wait),
                           ctypes.CFUNCTYPE(INT, ctypes.c_size_t)(lambda _: 2 if self.no_host_memory else 0))
        self.runtime.stand_in_connect(*self._callbacks)
        self.lib = ctypes.CDLL(LIBRARY)
        self.lib.ash_last_error.restype = ctypes.c_char_p
        self.ctr = None

    def kernels(self):
        name = self.runtime.stand_in_kernel
        name.restype = ctypes.c_char_p
        names = []
        while name(len(names)) is not None:
            names.append(name(len(names)).decode())
        return names

    def stream(self, number):
        return self.streams.setdefault(number, Stream())

    # ------------------------------------------------------- what the device does
    def _leave(self, landing, stamp, values):
        words = _words(landing)
        for w, value in enumerate(values):
            words[w] = (value & 0xFFFFFFFF) | ((stamp & 0xFFFFFFFF) << 32)

    def _change(self):
        if self.effects:
            for counter, by in self.effects.pop(0).items():
                self.ctr[counter] += by

    def _arg(self, args, k, layout):
        return struct.unpack(layout, ctypes.string_at(args[k], struct.calcsize(layout)))

    def _work(self, name, args, stream):
        """What the launch does, with its arguments as they are now."""
        arg = lambda k, layout: self._arg(args, k, layout)
        if "publish_counters_kernel" in name:
            (landing,), (stamp,) = arg(1, "<Q"), arg(2, "<i")
            return lambda: self._leave(landing, stamp, list(self.ctr)[:HOST_COUNTERS])
        if "set_counter_kernel" in name:
            (ctr,), (which,), (value,) = arg(0, "<Q"), arg(1, "<i"), arg(2, "<i")

            def store():
                ctypes.c_int32.from_address(ctr + 4 * which).value = value

            return store
        if "clear_kernel" in name or "reset_heap_kernel" in name:
            at = 1 if "clear_kernel" in name else 2
            (ctr,) = arg(at, "<Q")
            zero = "reset_heap_kernel" in name or arg(2, "<i")[0] != 0
            size = 0 if "clear_kernel" in name else arg(3, "<i")[0]

            def reset():
                if zero:
                    ctypes.memset(ctr, 0, 4 * HOST_COUNTERS)
                    self.ctr[SIZE] = size

            return reset
        publish = check = None
        if "insert_kernel" in name:
            publish, check = arg(6, "<QiiQ"), arg(7, "<IIQiiQ")
        elif "erase_kernel" in name:
            publish = arg(3, "<QiiQ")
        elif "insert_selected_kernel" in name:
            publish = arg(5, "<QiiQ")
        changes = (publish is not None or "activate" in name or "build_kernel" in name
                   or "erase_range_kernel" in name or "replace_from_log" in name)
        if "insert_selected_kernel" in name:
            changes = False      # (the build pass stands for the whole insert)
        early = None
        if "split_once_kernel" in name or "split_keys_kernel" in name:
            early = arg(4, "<Q") + arg(5, "<i")
        count = None
        if "count_flags_kernel" in name:
            count = arg(4, "<Q") + arg(5, "<i")

        owed = [publish and publish[0], early and early[0], count and count[0], check and check[0] and check[2]]
        self.words += [(stream, word) for word in owed if word]

        def work():
            if check is not None and check[0]:
                self._leave(check[2], check[3], [self.bad_keys])
            if early is not None and early[0]:
                self._leave(early[0], early[1], [self.spilled])
            if changes:
                self._change()
            if count is not None:
                self._leave(count[0], count[1], list(self.ctr)[:HOST_COUNTERS])
            if publish is not None and publish[0]:
                self._leave(publish[0], publish[1], list(self.ctr)[:HOST_COUNTERS])

        return work

    def _launch(self, name, stream, args):
        try:
            name = name.decode()
            for part in [p for p in self.before if p in name]:
                self.before.pop(part)()
            if any(part in name for part in self.refuse):
                return 98
            self.launched.append(name)
            queue = self.stream(stream)
            work = self._work(name, args, stream)
            if queue.held:
                queue.queue.append(work)
            else:
                work()
            return 0
        except BaseException:
            import traceback

            traceback.print_exc()
            os._exit(3)

    def _wait(self, stream):   # (a stream that is held is let go by whoever holds it)
        held = list(self.streams.values()) if stream == 2**64 - 1 else [self.stream(stream)]
        while any(s.held for s in held):
            time.sleep(0.001)
        return 0


class Map:
    def __init__(self, device, capacity=100_000, key_dim=3):
        self.device, self.lib, self.capacity = device, device.lib, capacity
        table, general = I64(), I64()
        self.ok(self.lib.ash_map_workspace_bytes(INT(key_dim), I64(capacity), ctypes.byref(table), ctypes.byref(general)))
        self._memory = [ctypes.create_string_buffer(n + 256) for n in (table.value, 4 * capacity, 20 << 16)]
        self.table, self.heap, self.general = (-(-ctypes.addressof(m) // 256) * 256 for m in self._memory)
        device.ctr = (I32 * 64).from_address(self.table)
        self.handle = PTR()
        self.ok(self.lib.ash_map_create(INT(key_dim), I64(capacity), PTR(self.heap), PTR(self.table), table, INT(0),
                                        PTR(0), ctypes.byref(self.handle)))

    def ok(self, status):
        assert status == 0, (status, self.lib.ash_last_error())

    def _aligned(self, size):
        self._memory.append(ctypes.create_string_buffer(size + 256))
        return PTR(-(-ctypes.addressof(self._memory[-1]) // 256) * 256)

    def keys(self):
        return PTR(4096)   # (nothing reads them)

    def insert(self, n=100, policy=EARLY, stream=0, values=0, row_bytes=16):
        need = I64()
        rows, nulls = (I64 * 4)(*[row_bytes] * 4), (PTR * 4)(4096, 4096, 4096, 4096)
        self.ok(self.lib.ash_map_insert_scratch_bytes(self.handle, I64(n), INT(values), rows, INT(policy),
                                                      ctypes.byref(need)))
        return self.lib.ash_map_insert_auto(self.handle, self.keys(), I64(n), INT(values), nulls, nulls, rows,
                                            self._aligned(need.value), need, INT(policy), PTR(0), PTR(stream))

    def erase(self, n=100, stream=0):
        return self.lib.ash_map_erase(self.handle, self.keys(), I64(n), PTR(stream))

    def activate(self, stream=0):
        return self.lib.ash_grid_activate_positions(
            self.handle, self.keys(), I64(10), PTR(0), ctypes.c_float(1.0), INT(8), INT(1), INT(1), INT(-100),
            INT(100), PTR(4096), PTR(4096), PTR(stream))

    def clear(self, stream=0):
        return self.lib.ash_map_clear(self.handle, PTR(stream))

    def attach(self, stream=0):
        return self.lib.ash_map_attach_general(self.handle, PTR(self.general), I64(19 << 16), PTR(stream))

    def size(self, stream=0):
        out = I64()
        self.ok(self.lib.ash_map_size(self.handle, ctypes.byref(out), PTR(stream)))
        return out.value

    def load(self, n, stream=0):
        return self.lib.ash_map_load(self.handle, self.keys(), PTR(4096), I64(n), PTR(self.heap), PTR(stream))

    def rebuild(self, stream=0):
        return self.lib.ash_map_rebuild(self.handle, PTR(4096), PTR(4096), I64(0), PTR(stream))

    def counters(self, stream=0):
        out = (I64 * 7)()
        self.ok(self.lib.ash_map_counters(self.handle, PTR(0), out, PTR(stream)))
        return list(out)

    def status(self, stream=0):
        out = (I64 * 5)()
        self.ok(self.lib.ash_map_status(self.handle, out, PTR(stream)))
        return out[0]

    def erase_bulk(self, n=100_000, stream=0):
        need, worth = I64(), INT()
        self.ok(self.lib.ash_map_erase_bulk_query(self.handle, I64(n), ctypes.byref(need), ctypes.byref(worth)))
        return self.lib.ash_map_erase_bulk(self.handle, self.keys(), I64(n), self._aligned(need.value), need,
                                           PTR(stream))

    def fuse(self, stream=0):
        f = ctypes.c_float
        return self.lib.ash_grid_fuse_frame(
            self.handle, self.keys(), I64(10), PTR(0), f(1.0), INT(1), INT(1), INT(-100), INT(100), PTR(4096),
            PTR(4096), PTR(4096), I64(self.capacity), INT(8), INT(5), f(1.0), PTR(0), PTR(4096), PTR(4096),
            PTR(4096), PTR(4096), INT(480), INT(640), f(0.1), f(4.0), PTR(4096), PTR(stream))

    def pending(self):
        return self.lib.ash_map_counters_pending(self.handle)


def beside(work):
    """`work()` in a thread of its own; `.result` once it is joined."""

    class Beside(threading.Thread):
        result = None

        def run(self):
            self.result = work()

    thread = Beside(daemon=True)
    thread.start()
    return thread


if __name__ == "__main__":
    import faulthandler

    faulthandler.dump_traceback_later(90, exit=True)
    import host_scenarios

    getattr(host_scenarios, sys.argv[2])(Device(sys.argv[1]))
    print("as it should be", flush=True)
    os._exit(0)
