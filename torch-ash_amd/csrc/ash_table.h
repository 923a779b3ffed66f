// Device-side helpers shared by the table kernels of libash_hip.so: key codec,
// hash, bucket addressing, the value-row descriptor of a fused insert.
#pragma once

#include "ash_dev.h"

namespace ash {

constexpr int kMaxFusedValues = 4;
constexpr int kMaxFusedRowDwords = 16;

// ------------------------------------------------------------ key codec
template <int DIM>
__device__ __forceinline__ bool pack_key(const int32_t (&k)[DIM],
                                         uint64_t& code) {
    if constexpr (DIM == 1) {
        code = static_cast<uint32_t>(k[0]);
        return true;
    } else if constexpr (DIM == 2) {
        const uint32_t u0 = static_cast<uint32_t>(k[0]) ^ 0x80000000u;
        const uint32_t u1 = static_cast<uint32_t>(k[1]) ^ 0x80000000u;
        code = static_cast<uint64_t>(u0) | (static_cast<uint64_t>(u1) << 32);
        return code < kTomb;
    } else if constexpr (DIM == 3) {
        const uint32_t u0 = static_cast<uint32_t>(k[0]) + (1u << 20);
        const uint32_t u1 = static_cast<uint32_t>(k[1]) + (1u << 20);
        const uint32_t u2 = static_cast<uint32_t>(k[2]) + (1u << 20);
        code = static_cast<uint64_t>(u0) | (static_cast<uint64_t>(u1) << 21) |
               (static_cast<uint64_t>(u2) << 42);
        return (u0 | u1 | u2) < (1u << 21);
    } else {
        const uint32_t u0 = static_cast<uint32_t>(k[0]) + 32768u;
        const uint32_t u1 = static_cast<uint32_t>(k[1]) + 32768u;
        const uint32_t u2 = static_cast<uint32_t>(k[2]) + 32768u;
        const uint32_t u3 = static_cast<uint32_t>(k[3]) + 32768u;
        code = static_cast<uint64_t>(u0) | (static_cast<uint64_t>(u1) << 16) |
               (static_cast<uint64_t>(u2) << 32) |
               (static_cast<uint64_t>(u3) << 48);
        return (u0 | u1 | u2 | u3) < 65536u && code < kTomb;
    }
}

template <int DIM>
__device__ __forceinline__ void unpack_key(uint64_t code, int32_t (&k)[DIM]) {
    if constexpr (DIM == 1) {
        k[0] = static_cast<int32_t>(static_cast<uint32_t>(code));
    } else if constexpr (DIM == 2) {
        k[0] = static_cast<int32_t>(static_cast<uint32_t>(code) ^ 0x80000000u);
        k[1] = static_cast<int32_t>(static_cast<uint32_t>(code >> 32) ^
                                    0x80000000u);
    } else if constexpr (DIM == 3) {
        k[0] = static_cast<int32_t>(code & 0x1FFFFFu) - (1 << 20);
        k[1] = static_cast<int32_t>((code >> 21) & 0x1FFFFFu) - (1 << 20);
        k[2] = static_cast<int32_t>((code >> 42) & 0x1FFFFFu) - (1 << 20);
    } else {
        k[0] = static_cast<int32_t>(code & 0xFFFFu) - 32768;
        k[1] = static_cast<int32_t>((code >> 16) & 0xFFFFu) - 32768;
        k[2] = static_cast<int32_t>((code >> 32) & 0xFFFFu) - 32768;
        k[3] = static_cast<int32_t>((code >> 48) & 0xFFFFu) - 32768;
    }
}

__device__ __forceinline__ uint64_t mix64(uint64_t h) {
    h ^= h >> 33;
    h *= 0xff51afd7ed558ccdull;
    h ^= h >> 33;
    h *= 0xc4ceb9fe1a85ec53ull;
    h ^= h >> 33;
    return h;
}

__device__ __forceinline__ uint32_t bucket_of(uint64_t code, uint32_t nb) {
    return __umulhi(static_cast<uint32_t>(mix64(code) >> 32), nb);
}

// The slot of a bucket that a new key tries first; the others follow, around the bucket.
// Keys of a batch that meet in a bucket claim different slots that way, where all of them
// went for the first free one and then, but for one, for the next: a trip to where atomics
// are done each time, and four keys a bucket are what a filling map has (the kernel alone,
// us: 100 000 keys with rows into an emptied map 23.3 -> 17.4, 200 000 33.4 -> 23.5, keys
// alone 20.0 -> 15.7; beside 47 000 keys 190 000 43 -> 32, 300 000 51 -> 38.7; beside a
// million 65 537 15.7 -> 15.4, 300 000 33.4 -> 30.9).
__device__ __forceinline__ int first_slot(uint64_t code) {
    return static_cast<int>(__umulhi(static_cast<uint32_t>(mix64(code)), static_cast<uint32_t>(kSlots)));
}

// The bucket after b in b's probe sequence: the next one of b's aligned range
// of kPartBuckets buckets, wrapping inside that range (a table of fewer
// buckets is one shorter range).  A sequence visits at most kPartBuckets buckets.
__device__ __forceinline__ uint32_t next_bucket(uint32_t b, uint32_t nb) {
    const uint32_t n = b + 1;
    return ((n & (kPartBuckets - 1)) == 0 || n == nb) ? (b & ~(kPartBuckets - 1)) : n;
}

template <int DIM>
__device__ __forceinline__ void load_key(const int32_t* __restrict__ keys,
                                         int64_t i, bool active,
                                         int32_t (&k)[DIM]) {
#pragma unroll
    for (int d = 0; d < DIM; ++d) k[d] = active ? keys[i * DIM + d] : 0;
}

// The same for keys that are read once and come from memory, marked as not to be kept
// in the caches: what is written meanwhile stays there instead.
template <int DIM>
__device__ __forceinline__ void load_key_once(const int32_t* __restrict__ keys, int64_t i,
                                              int32_t (&k)[DIM]) {
#pragma unroll
    for (int d = 0; d < DIM; ++d) k[d] = __builtin_nontemporal_load(keys + i * DIM + d);
}

// Value rows copied by a fused insert: row i of src[v] goes to row `index` of
// dst[v]; rows are row_dwords[v] 32-bit words long.
struct ValueArgs {
    int n;
    const uint32_t* src[kMaxFusedValues];
    uint32_t* dst[kMaxFusedValues];
    int32_t row_dwords[kMaxFusedValues];
};

// ---------------------------------------------------------------- host
struct DeviceGuard {
    int prev = -1;
    bool switched = false;
    hipError_t enter(int device) {
        hipError_t e = hipGetDevice(&prev);
        if (e != hipSuccess) return e;
        if (prev != device) {
            e = hipSetDevice(device);
            switched = (e == hipSuccess);
        }
        return e;
    }
    ~DeviceGuard() {
        if (switched) (void)hipSetDevice(prev);
    }
};

// The entry points that take tensors but no map (queries, convolution, surface
// extraction, depth integration) run on the device that holds their first
// tensor: the runtime is asked where the pointer lives and that device is made
// current for the call.  A pointer the runtime does not know leaves the
// current device as it is.
struct PointerGuard : DeviceGuard {
    hipError_t enter_for(const void* p) {
        if (p == nullptr) return hipSuccess;
        hipPointerAttribute_t attr;
        if (hipPointerGetAttributes(&attr, p) != hipSuccess) {
            (void)hipGetLastError();
            return hipSuccess;
        }
        if (attr.type != hipMemoryTypeDevice) return hipSuccess;
        return enter(attr.device);
    }
};

// Inserts the keys selected by `sel[0 .. *nsel)` (both on the device) with the
// per-key atomic kernel.  `codes` false: `keys` are int32[.., key_dim] rows and
// sel holds row numbers; true: `keys` are packed 64-bit codes.  The value rows
// of va.src are addressed by the same selected row number.  Defined in
// ash_map.hip.
// `publish`: what the last launch of a call leaves for the host, see
// publish_counters_kernel; `ticket` (zero) counts its workgroups.
struct Publish {
    uint64_t* landing;   // null: nothing
    int32_t stamp;
    int32_t* ticket;
};
int insert_selected(ash_map* map, bool codes, const void* keys,
                    const int32_t* sel, const int32_t* nsel,
                    const ValueArgs& va, hipStream_t s,
                    const Publish& publish = {});

// Erases the selected keys with the per-key kernel; arguments as for
// insert_selected.
int erase_selected(ash_map* map, bool codes, const void* keys, const int32_t* sel,
                   const int32_t* nsel, hipStream_t s);

int check_batch(const ash_map* map, const void* keys, int64_t n);
// The value tables of an insert.
int check_rows(int n_values, const void* const* src, void* const* dst, const int64_t* row_bytes);
inline bool is_capturing(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

// A place among the counters for a launch whose workgroups count themselves.  Launches
// on one stream could share one; as many as there are places may run at a time on
// several (a captured launch keeps its own).
inline int next_slot(ash_map* map) { return static_cast<int>(map->launches.fetch_add(1) % kLaunchSlots); }

// Whether the heap array is known to be 0, 1, 2, ...
inline bool heap_in_order(const ash_map* map) { return !map->heap_dirty && !map->replayed; }

// A call that changes the counters, from before its first launch until its last is
// queued (at the latest when it is left): at both ends what the host keeps of them
// lapses, since what a reader has asked for in between may be from before.
enum ChangeKind {
    kChangeAdds,     // may have added entries (and ends without a look at the counters)
    kChangeErases,   // may have left tombstones
    kChangeElse
};

class Change {
  public:
    // `s`: the stream the call runs on (where one that adds or erases is captured, see
    // ash_map::replayed)
    Change(ash_map* map, ChangeKind kind, hipStream_t s);
    Change(const Change&) = delete;
    Change& operator=(const Change&) = delete;
    ~Change() { queued(); }
    void queued();
    void queued_with(const ash_counters& c);   // ... and has left the counters at `c`

  private:
    void lapse();   // the caller holds the map's counter_lock
    ash_map* map_;
};
// Leaves `value` for the host in a word of its line (kLineWords).
__device__ __forceinline__ void leave_word(uint64_t* word, int32_t value, int32_t stamp) {
    __hip_atomic_store(word, static_cast<uint64_t>(static_cast<uint32_t>(value)) |
                                     (static_cast<uint64_t>(static_cast<uint32_t>(stamp)) << 32),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
inline int32_t value_of(uint64_t word) { return static_cast<int32_t>(static_cast<uint32_t>(word)); }
inline int32_t stamp_of(uint64_t word) { return static_cast<int32_t>(static_cast<uint32_t>(word >> 32)); }

// Page-locked words of one call's own, in which a kernel leaves what the call
// waits for, each under the call's stamp.
class Answer {
  public:
    Answer() = default;
    Answer(const Answer&) = delete;
    Answer& operator=(const Answer&) = delete;
    ~Answer();
    int take();                // `words` and `stamp` are the call's from here on
    // `s`: the stream whose latest launch leaves the first `count` words
    int wait(hipStream_t s, int count);
    int64_t pair(int w) const {   // words w (below) and w + 1
        return static_cast<int64_t>(static_cast<uint32_t>(value_of(words[w]))) |
               (static_cast<int64_t>(value_of(words[w + 1])) << 32);
    }
    void abandon() { lost_ = true; }   // nobody waits for words that may still come
    uint64_t* words = nullptr;
    int32_t stamp = 0;

  private:
    bool lost_ = false;   // the device may still owe the words
};
// The map's own page-locked words (made on first use), and the wait for some of them.
int take_line(ash_map* map);
int wait_for_words(const uint64_t* words, int count, int32_t stamp);
// May the table hold tombstones, for an insert?  (Replays of a captured launch meet
// any table; refused keys whose counters nobody has read yet may have left some,
// which then wait for a later insert.)
inline bool tombs_in(const ash_map* map) { return map->maybe_tombstones || map->replayed; }
// Counts the flags that are up among the first `rows` into the counter of touched
// blocks and queues the read-back of the counters behind the stream's work; `counts`:
// `max_counts` words of scratch on the device (ash_map.hip).
int queue_touched_count(ash_map* map, const uint8_t* touched, int64_t rows, int32_t* counts,
                        int max_counts, hipStream_t s);
// The streaming insert (ash_bulk.hip); `early`: page-locked word (or null) where
// its first pass leaves the number of keys that it hands to the per-key kernel,
// under `stamp`.  With `early` the call waits for that number; is it zero, the last
// launch leaves the counters at `late` (under `stamp`) and *published is set.
int insert_bulk(ash_map* map, const int32_t* keys, int64_t n, int n_values,
                const void* const* src, void* const* dst, const int64_t* row_bytes,
                void* workspace, int64_t workspace_bytes, uint64_t* early, uint64_t* late,
                int32_t stamp, bool* published, void* stream);
// Whether a batch is one to stream under ASH_STREAMING_EARLY (ash_bulk.hip).
bool streams_early(const ash_map* map, int64_t n, int n_values);
// Buckets up to which a clear fills the table at once, in the launch that resets the
// counters (2.8 MB, half a microsecond of stores where a streaming insert follows).
constexpr int64_t kFillAtOnce = 21845;
// Fills the bucket array if a clear() left that to the next user of the table.
int settle_table(ash_map* map, hipStream_t s);
// Before the first call that writes to the heap (an erase; a load brings a
// heap of its own): from here on items() reads the whole key log, so what a
// clear() left in it beyond the size is emptied now.
int give_up_heap_order(ash_map* map, hipStream_t s);

}  // namespace ash
