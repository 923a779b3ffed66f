// Hash map of libash_hip.so: a bucketed open-addressing table for gfx950.
//
// Layout.  A bucket is one 128-byte line holding ten 64-bit key codes followed
// by their ten int32 indices, so a lookup that hits touches one line.  A key
// int32[dim] is packed into a 64-bit code (dim 1: 32 bits, dim 2: 2x32 biased,
// dim 3: 3x21 biased, dim 4: 4x16 biased); a slot is claimed with one 64-bit
// compare-and-swap of the code, which is also what makes duplicate keys inside
// one batch collapse without locks.  Keys whose components do not fit the code
// ("exotic" keys) live in a second, lock-based open-addressing region that is
// only attached once such a key shows up.
//
// Probing.  A wavefront takes 64 keys.  Each quad of lanes owns four of them
// and probes them one after the other: the four lanes read the 128 bytes of
// the key's bucket in two coalesced requests, compare, and agree through quad
// permutations.  All reads of a quad are issued before the first compare, so a
// wavefront keeps 64 lines in flight.  If the bucket neither holds the key
// nor an empty slot the key moves on to the next bucket.
//
// Index allocation follows the reference's heap protocol
// (ash/src/hashmap_gpu.cuh:211-232,316-336): a new key takes heap[counter++],
// an erased key stores its index at heap[--counter]; here the counter is
// advanced once per workgroup instead of once per key.
#include "ash_probe.h"
#include "ash_walk.h"

#include "../../include/ash_hip.h"

#include <hip/amd_detail/amd_hip_unsafe_atomics.h>

#include <algorithm>
#include <chrono>
#include <cstring>
#include <mutex>
#include <thread>
#include <type_traits>
#include <vector>

// Scratch of ash_grid_activate_static, the entry point that allocates nothing:
// the list of run heads that ash_grid_activate keeps in a caller-provided
// temporary (one counter line + three int32 per position).  Every device that
// loads the library holds its own copy until the process ends.  In host code
// this name is only a handle for hipGetSymbolAddress; kernels are given the
// address that call returned for the current device.
constexpr int64_t kActivateStaticMax = ASH_ACTIVATE_STATIC_MAX_POSITIONS;
static __device__ __align__(256) int32_t scratch[64 + 3 * kActivateStaticMax];

namespace ash {

static thread_local std::string g_last_error;
void set_error(const std::string& msg) { g_last_error = msg; }

namespace {

constexpr int kBlock = 256;
// Workgroup size of the kernels that advance the heap counter (once per
// workgroup).  Larger groups mean fewer updates of that single address but make
// every wavefront wait for the slowest probe of the group (kWideInsert).
constexpr int kHeapBlock = 256;
constexpr uint32_t kSpinLimit = 1u << 22;

// -------------------------------------------------- cooperative probe pass
enum { kProbeFound = 0, kProbeHasEmpty = 1, kProbeFull = 2 };

struct ProbeResult {
    int status;      // kProbe*
    int slot;        // matching slot (status == kProbeFound)
    int32_t val;     // index stored with the matching slot
    uint32_t emask;  // bit s set <=> slot s was empty in this snapshot
    uint32_t tmask;  // ... held a tombstone (asked for with TOMBS)
};

// Every lane of the wavefront calls this together.  Lane L owns key L; in
// round r the four lanes of a quad read the bucket `b` of the quad's r-th key
// (two 16-byte pieces per lane: codes 0..7 with the first, codes 8, 9 and the
// ten indices with the second) and the result lands in that key's owner lane.
// Keys that are not pending cost no memory traffic.
// A quad, because what its lanes tell each other -- whose key, which slot,
// which index -- are quad permutations, modifiers of a vector instruction, where
// groups of eight have to go through ballots and the LDS pipeline.
template <bool TOMBS = false>
__device__ __forceinline__ void probe_pass(const MapDev& m, uint64_t code,
                                           uint32_t b, bool pend, int lane,
                                           ProbeResult& out) {
    static_assert(kSlots == 10 && kBucketDwords == 32, "two 16-byte pieces per lane");
    const int j = lane & 3;
    uint4 lo[4], hi[4];
    auto fetch = [&](auto round) {
        constexpr int r = decltype(round)::value;
        const uint32_t br = quad_bcast<r>(b);
        lo[r] = make_uint4(0u, 0u, 0u, 0u);
        hi[r] = make_uint4(0u, 0u, 0u, 0u);
        if (quad_bcast<r>(pend ? 1u : 0u)) {
            const uint4* line = reinterpret_cast<const uint4*>(
                    m.buckets + static_cast<size_t>(br) * kBucketQwords);
            lo[r] = line[j];
            hi[r] = line[4 + j];
        }
    };
    auto compare = [&](auto round) {
        constexpr int r = decltype(round)::value;
        const uint64_t want = static_cast<uint64_t>(quad_bcast<r>(static_cast<uint32_t>(code))) |
                              (static_cast<uint64_t>(quad_bcast<r>(static_cast<uint32_t>(code >> 32))) << 32);
        const uint64_t q0 = lo[r].x | (static_cast<uint64_t>(lo[r].y) << 32);
        const uint64_t q1 = lo[r].z | (static_cast<uint64_t>(lo[r].w) << 32);
        // (codes 8 and 9, in the quad's first lane; indices in the others)
        const uint64_t q8 = j == 0 ? hi[r].x | (static_cast<uint64_t>(hi[r].y) << 32) : 0ull;
        const uint64_t q9 = j == 0 ? hi[r].z | (static_cast<uint64_t>(hi[r].w) << 32) : 0ull;
        uint32_t v = 0;   // bits 0..3: slot + 1 of the match, 4..13: empty slots, 14..23: tombstones
        if (j == 0 && q8 == want) v = 9;
        if (j == 0 && q9 == want) v = 10;
        if (q0 == want) v = 2 * j + 1;
        if (q1 == want) v = 2 * j + 2;
        if (q0 == kEmpty) v |= 16u << (2 * j);
        if (q1 == kEmpty) v |= 32u << (2 * j);
        if (q8 == kEmpty) v |= 16u << 8;
        if (q9 == kEmpty) v |= 16u << 9;
        if constexpr (TOMBS) {
            if (q0 == kTomb) v |= 16384u << (2 * j);
            if (q1 == kTomb) v |= 32768u << (2 * j);
            if (q8 == kTomb) v |= 16384u << 8;
            if (q9 == kTomb) v |= 16384u << 9;
        }
        v = quad_or(v);
        const int slot = static_cast<int>(v & 15u) - 1;
        const int comp = slot & 3;   // index of slot s: dword 20 + s of the bucket
        const uint32_t word = comp == 0 ? hi[r].x : comp == 1 ? hi[r].y : comp == 2 ? hi[r].z : hi[r].w;
        const uint32_t val = quad_or(j == ((4 + slot) >> 2) ? word : 0u);
        if (j == r) {
            out.emask = (v >> 4) & ((1u << kSlots) - 1u);
            if constexpr (TOMBS) out.tmask = v >> (4 + kSlots);
            out.status = slot >= 0 ? kProbeFound : (out.emask ? kProbeHasEmpty : kProbeFull);
            out.slot = slot;
            out.val = static_cast<int32_t>(val);
        }
    };
    fetch(Round<0>());
    fetch(Round<1>());
    fetch(Round<2>());
    fetch(Round<3>());
    compare(Round<0>());
    compare(Round<1>());
    compare(Round<2>());
    compare(Round<3>());
}

// The same by every lane for itself (see kAloneKeys), and with no answer for keys that
// are not pending.  VAL: the index is asked for as well, along with the codes: read
// behind them, the line has often gone to an atomic of another lane in between (erases
// of 131 000 keys 13.4 -> 15.6 us when it was).
template <bool TOMBS = false, bool VAL = true>
__device__ __forceinline__ void probe_alone(const MapDev& m, uint64_t code, uint32_t b, bool pend,
                                            ProbeResult& out) {
    if (!pend) return;
    constexpr int kPieces = VAL ? kGroup : kSlots / 2;
    const uint4* line = reinterpret_cast<const uint4*>(m.buckets + static_cast<size_t>(b) * kBucketQwords);
    uint4 w[kPieces];
#pragma unroll
    for (int r = 0; r < kPieces; ++r) w[r] = line[r];
    out.slot = -1;
    out.emask = 0;
    if constexpr (TOMBS) out.tmask = 0;
    if constexpr (VAL) out.val = 0;
#pragma unroll
    for (int s = kSlots - 1; s >= 0; --s) {
        const uint4 v = w[s / 2];
        const uint64_t q = s % 2 == 0 ? v.x | (static_cast<uint64_t>(v.y) << 32)
                                      : v.z | (static_cast<uint64_t>(v.w) << 32);
        if (q == code) out.slot = s;
        if constexpr (VAL) {
            static_assert(kValDword0 % 4 == 0, "four indices to a piece");
            const uint4 i = w[(kValDword0 + s) / 4];
            const uint32_t val = s % 4 == 0 ? i.x : s % 4 == 1 ? i.y : s % 4 == 2 ? i.z : i.w;
            if (q == code) out.val = static_cast<int32_t>(val);
        }
        if (q == kEmpty) out.emask |= 1u << s;
        if constexpr (TOMBS) {
            if (q == kTomb) out.tmask |= 1u << s;
        }
    }
    out.status = out.slot >= 0 ? kProbeFound : (out.emask ? kProbeHasEmpty : kProbeFull);
}

// ------------------------------------------------ general (exotic) region
enum { kGenWon = 0, kGenDup = 1, kGenFull = 2, kGenNoRegion = 3 };

// Claims a slot for an exotic key.  The slot word goes EMPTY -> LOCKED ->
// NOINDEX (key readable); the caller later stores the index.  A thread that
// meets LOCKED re-reads the word; the holder finishes its few stores inside
// the same loop trip, and the wait is bounded by kSpinLimit.
template <int DIM>
__device__ int gen_claim(const MapDev& m, const int32_t (&k)[DIM],
                         uint32_t& pos) {
    if (m.gstate == nullptr) return kGenNoRegion;
    const uint32_t mask = m.gslots - 1;
    uint32_t p = gen_home<DIM>(k, m.gslots);
    uint32_t step = 0;
    uint32_t spins = 0;
    int result = kGenFull;
    bool done = false;
    while (!done) {
        int32_t w = gen_load(m.gstate + p);
        if (w == kGenEmpty) {
            const int32_t old = atomicCAS(m.gstate + p, kGenEmpty, kGenLocked);
            if (old == kGenEmpty) {
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    __hip_atomic_store(
                            m.gkeys + static_cast<size_t>(p) * 4 + d,
                            d < DIM ? k[d < DIM ? d : 0] : 0, __ATOMIC_RELAXED,
                            __HIP_MEMORY_SCOPE_AGENT);
                }
                __hip_atomic_store(m.gstate + p, kGenNoIndex, __ATOMIC_RELEASE,
                                   __HIP_MEMORY_SCOPE_AGENT);
                pos = p;
                result = kGenWon;
                done = true;
                w = kGenNoIndex;
            } else {
                w = old;
            }
        }
        if (!done) {
            if (w == kGenLocked) {
                if (++spins >= kSpinLimit) done = true;  // give up: kGenFull
            } else {
                if (w != kGenTomb && w != kGenEmpty) {
                    __atomic_thread_fence(__ATOMIC_ACQUIRE);
                    if (gen_key_equal<DIM>(m, p, k)) {
                        result = kGenDup;
                        done = true;
                    }
                }
                if (!done && w != kGenEmpty) {
                    p = (p + 1) & mask;
                    if (++step >= m.gslots) done = true;
                }
            }
        }
    }
    return result;
}

// ------------------------------------------------------------- kernels
// Looks key `k` up; every lane of the wavefront calls this together, lanes
// with active == false only help.  Returns whether the key is stored and, if
// so, its index in `res`.
template <int DIM>
__device__ __forceinline__ bool find_key(const MapDev& m, const int32_t (&k)[DIM],
                                         bool active, int32_t& res) {
    const int lane = threadIdx.x & 63;
    uint64_t code;
    const bool fits = pack_key<DIM>(k, code);
    bool pend = active && fits;
    uint32_t b = bucket_of(code, m.nb);
    uint32_t steps = 0;
    res = 0;
    bool found = false;
    while (__ballot(pend)) {
        ProbeResult p;
        probe_pass(m, code, b, pend, lane, p);
        if (pend) {
            if (p.status == kProbeFound) {
                found = true;
                res = p.val;
                pend = false;
            } else if (p.status == kProbeHasEmpty) {
                pend = false;
            } else {
                b = next_bucket(b, m.nb);
                if (++steps >= kPartBuckets) pend = false;
            }
        }
    }
    if (active && !fits) {
        uint32_t pos;
        found = gen_find<DIM>(m, k, res, pos);
    }
    return found;
}

// Keys up to which every lane looks its own up (find_key_alone): half the vector
// instructions and registers, and one trip to memory less before the codes are
// compared, but five requests per line instead of two, which bound batches that fill the
// device.  A batch, cooperative -> alone (us): without rows, among a million keys 131 000
// 7.5 -> 6.6, 300 000 10.8 -> 8.6, 500 000 15.3 -> 12.5, 1 M 23.9 -> 21.9, among 100 000
// 10.7 -> 9.8 at 500 000, 12.3 -> 12.5 at 700 000, 15.6 -> 16.9 at 1 M, 85 -> 113 at 8 M;
// with rows of 12 and 4 bytes 131 000 10.2 -> 9.4, 200 000 12.1 -> 11.6, 300 000 14.5
// -> 14.7, 1 M 41 -> 44.  Up to the bounds the size of the table does not matter: among four
// million | sixteen, of which seven in ten are stored, 2^19 16.3 -> 13.7 | 17.9 -> 15.9, with
// rows 2^18 14.9 -> 15.2 | 15.6 -> 15.3 (all stored 17.1 -> 17.4 | 18.8 -> 19.5, none 13.8
// -> 9.9 | 13.5 -> 10.2).
constexpr int64_t kAloneKeys = int64_t{1} << 19, kAloneKeysWithRows = int64_t{1} << 18;

template <int DIM, bool ALONE>
__device__ __forceinline__ bool look_up(const MapDev& m, const int32_t (&k)[DIM], bool active, int32_t& res) {
    if constexpr (ALONE) return find_key_alone<DIM>(m, k, active, res);
    else return find_key<DIM>(m, k, active, res);
}

template <int DIM, bool ALONE>
__global__ __launch_bounds__(kBlock) void find_kernel(
        MapDev m, const int32_t* __restrict__ keys, int64_t n,
        int64_t* __restrict__ idx_out, uint8_t* __restrict__ mask_out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    const bool active = i < n;
    int32_t k[DIM];
    load_key<DIM>(keys, i, active, k);
    int32_t res = 0;
    const bool found = look_up<DIM, ALONE>(m, k, active, res);
    if (active) {
        idx_out[i] = found ? static_cast<int64_t>(res) : 0;
        mask_out[i] = found ? 1 : 0;
    }
}

// Fused front end of the sparse-dense grid query (ash/grid.py:183-199): splits a
// position x (cell units) into block / cell / fractional part (split_axis) and
// looks the block up (find_block_by_runs), in one pass.
__global__ __launch_bounds__(kBlock) void grid_query_kernel(
        MapDev m, const float* __restrict__ x, int64_t n, float g, int gi,
        int64_t* __restrict__ grid_idx, int64_t* __restrict__ cell_idx,
        float* __restrict__ off, uint8_t* __restrict__ mask_out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    const bool active = i < n;
    int32_t k[3];
    float o[3];
    int64_t cell = 0;
    int64_t stride = 1;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        int32_t c;
        split_axis(active ? x[i * 3 + d] : 0.f, g, k[d], c, o[d]);
        cell += static_cast<int64_t>(c) * stride;
        stride *= gi;
    }
    int32_t res = 0;
    const bool found = find_block_by_runs(m, k, active, res);
    if (active) {
        grid_idx[i] = found ? static_cast<int64_t>(res) : 0;
        mask_out[i] = found ? 1 : 0;
        cell_idx[i] = cell;
        off[i * 3 + 0] = o[0];
        off[i * 3 + 1] = o[1];
        off[i * 3 + 2] = o[2];
    }
}

enum InsertMode {
    kInsertKeys = 0,    // allocate indices only
    kInsertFused = 1,   // + copy narrow value rows in the same kernel
    kInsertAssign = 2,  // + report the allocated index per input row
    kInsertLoad = 3,    // indices are given (state-dict load), heap untouched
    kInsertReport = 4   // keys only; tells the caller the key's index when it is final
};

// A change of a counter by one thread, which has been made when this returns: the
// old value has come back from where the change is made.
__device__ __forceinline__ void change_counter(int32_t* counter, int32_t by) {
    const int32_t old = atomicAdd(counter, by);
    asm volatile("" ::"v"(old) : "memory");
}

// The size and the number of tombstones changed at once, which costs one place in the
// queue for their line instead of two (batches that come, are read and go, us: 65 537 beside
// a million 89.9 -> 88.2, 120 000 109.9 -> 103.8, 300 000 161.6 -> 156.4, a million beside
// four 397 -> 391); returns the size before.  What the lower half
// carries over is put back: a size below zero, or out of there, as refused loads may
// leave it.
__device__ __forceinline__ int32_t change_size(int32_t* ctr, int32_t by, int32_t tombs) {
    static_assert(kCtrSize % 2 == 0 && kCtrTombs == kCtrSize + 1, "two halves of a 64-bit word");
    const uint64_t delta = (static_cast<uint64_t>(static_cast<uint32_t>(tombs)) << 32) +
                           static_cast<uint64_t>(static_cast<int64_t>(by));
    const uint64_t old = atomicAdd(reinterpret_cast<unsigned long long*>(ctr + kCtrSize),
                                   static_cast<unsigned long long>(delta));
    const uint32_t before = static_cast<uint32_t>(old);
    const bool carry = before + static_cast<uint32_t>(by) < before;
    if (by > 0 && carry) change_counter(ctr + kCtrTombs, -1);
    if (by < 0 && !carry) change_counter(ctr + kCtrTombs, 1);
    return static_cast<int32_t>(before);
}

// The insert proper for a key held in registers (`code` is its packed form if
// `fits`); `i` is the row of the key's value rows / `assigned` / `given` entry.
// TOMBS: the table may hold tombstones (the same for the whole launch).
// BLOCK: threads of the workgroup, all of which call this together.  ALONE: buckets are
// looked at by each lane for itself.
template <int DIM, int MODE, bool TOMBS, int BLOCK = kHeapBlock, bool ALONE = false>
__device__ __forceinline__ void insert_key(
        const MapDev& m, const int32_t (&k)[DIM], uint64_t code, bool fits,
        int64_t i, bool active, const ValueArgs& va,
        int32_t* __restrict__ assigned, const int64_t* __restrict__ given,
        int32_t* report = nullptr) {
    static_assert(!(TOMBS && MODE == kInsertLoad), "loads start from an emptied table");
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    int32_t seen = -1;     // kInsertReport: the index read beside a key that was there
    bool gdup = false;     // kInsertReport: the key stands in the general region
    bool pend = active && fits;
    uint32_t b = bucket_of(code, m.nb);
    const int turn = first_slot(code);
    uint32_t steps = 0;

    bool won = false;      // claimed a packed slot (wb, ws)
    bool gwon = false;     // claimed a general slot gp
    bool refused = false;  // no room anywhere
    uint32_t wb = 0, gp = 0;
    int ws = 0;

    // Phase A: claim a slot per new key.  Its sequence is followed to the end (a bucket
    // with an empty slot, or the whole range): a key that is met there is stored
    // already.  Else it takes the first slot of the sequence that is free, empty or a
    // tombstone.  Slots are tried in the order of the sequence, so threads that store
    // the same key meet in the same slot, whatever others have taken in between --
    // unless a slot before it comes free meanwhile, which it does where a key finds
    // the heap exhausted and gives its slot back (phase B).  Whoever takes that one
    // has seen it free, and so draws from the heap after that key did: the counter
    // has reached the capacity, does not fall below it again in the same launch, and
    // the newcomer is refused as well.  Of two threads that store one key in two slots
    // at most one gets an index.
    // (Tombstones that are left alone pile up: keys that come and go behind a run of
    // full buckets lengthen it by what they leave each time, until the range is full
    // and refuses keys.  A million stored keys, 65 537 that come, are read and go:
    // 125 us a pass, but 1000 - 2700 after sixty passes on one map in twelve.)
    // One loop with one look at a bucket in it: with a second loop that starts over,
    // the kernel's instructions take their time to arrive (172 keys 6.9 -> 9.4 us,
    // 41 000 14.2 -> 16.2); hence the first tombstones met are kept until the end of
    // the sequence is (172 keys 7.5).  Without TOMBS (the host knows of none) nobody
    // looks for them, and the buckets on the way have nothing to take.
    bool claiming = false;   // the sequence has been followed to its end
    bool reused = false;
    uint32_t first_tombs = 0, first_b = 0, first_steps = 0;   // in a bucket on the way
    while (__ballot(pend)) {
        ProbeResult p;
        if constexpr (ALONE) probe_alone<TOMBS, MODE == kInsertReport>(m, code, b, pend, p);
        else probe_pass<TOMBS>(m, code, b, pend, lane, p);
        if (pend) {
            if (p.status == kProbeFound) {
                pend = false;
                if constexpr (MODE == kInsertLoad) {
                    atomicAdd(m.ctr + kCtrLoadDup, 1);
                }
                if constexpr (MODE == kInsertReport) seen = p.val;
            } else {
                uint32_t em = p.emask;   // (without TOMBS: of the sequence's last bucket)
                if constexpr (TOMBS) {
                    if (!claiming) {
                        if (first_tombs == 0) {
                            first_tombs = p.tmask;
                            first_b = b;
                            first_steps = steps;
                        }
                        claiming = p.status == kProbeHasEmpty || steps + 1 >= kPartBuckets;
                        if (claiming && first_tombs != 0 && first_steps != steps) {
                            p.emask = 0;
                            p.tmask = first_tombs;
                            b = first_b;
                            steps = first_steps;
                        }
                    }
                    em = claiming ? p.emask | p.tmask : 0u;
                }
                em = (em | (em << kSlots)) >> turn & ((1u << kSlots) - 1u);
                while (em) {
                    const int at = __builtin_ctz(em) + turn;
                    const int s = at < kSlots ? at : at - kSlots;
                    const unsigned long long free = TOMBS && ((p.tmask >> s) & 1u) ? kTomb : kEmpty;
                    const unsigned long long old = atomicCAS(slot_ptr(m, b, s), free, code);
                    if (old == free) {
                        won = true;
                        reused = free == kTomb;
                        wb = b;
                        ws = s;
                        pend = false;
                        break;
                    }
                    if (old == code) {
                        pend = false;
                        if constexpr (MODE == kInsertLoad) {
                            atomicAdd(m.ctr + kCtrLoadDup, 1);
                        }
                        break;
                    }
                    em &= em - 1;
                }
                if (pend) {
                    b = next_bucket(b, m.nb);
                    if (++steps >= kPartBuckets) {
                        pend = false;
                        refused = true;
                    }
                }
            }
        }
    }
    if (active && !fits) {
        const int g = gen_claim<DIM>(m, k, gp);
        if (g == kGenWon) {
            gwon = true;
        } else if (g == kGenFull) {
            refused = true;
        } else if (g == kGenNoRegion) {
            change_counter(m.ctr + kCtrExotic, 1);
        } else if constexpr (MODE == kInsertLoad) {
            atomicAdd(m.ctr + kCtrLoadDup, 1);
        } else if constexpr (MODE == kInsertReport) {
            gdup = true;
        }
    }
    if (refused) change_counter(m.ctr + kCtrDropped, 1);

    // Phase B: one heap-counter update per block, indices for the winners.
    const bool w = won || gwon;
    int32_t idx = -1;
    const int nreused = TOMBS ? __popcll(__ballot(reused)) : 0;
    if constexpr (MODE == kInsertLoad) {
        if (w) {
            // the index comes with the key (`given` null: the key's own number,
            // when the keys are the entries of the key log)
            const int64_t g = given != nullptr ? given[i] : i;
            if (g >= 0 && g < m.capacity) {
                idx = static_cast<int32_t>(g);
            } else {
                // an index that addresses no row: the pair is refused (the
                // slot goes back) and counted with the duplicates
                if (won) {
                    atomicExch(slot_ptr(m, wb, ws), kTomb);
                } else {
                    __hip_atomic_store(m.gstate + gp, kGenTomb, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                    atomicAdd(m.ctr + kCtrGenTombs, 1);
                }
                atomicAdd(m.ctr + kCtrTombs, 1);
                atomicAdd(m.ctr + kCtrLoadDup, 1);
            }
        }
    } else {
        __shared__ int s_cnt[BLOCK / 64];
        __shared__ int s_reused[BLOCK / 64];
        __shared__ int s_base;
        const uint64_t wm = __ballot(w);
        const int nw = __popcll(wm);
        const int rank = __popcll(wm & ((1ull << lane) - 1ull));
        if (lane == 0) {
            s_cnt[wave] = nw;
            if constexpr (TOMBS) s_reused[wave] = nreused;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            int tot = 0, again = 0;
#pragma unroll
            for (int q = 0; q < BLOCK / 64; ++q) {
                tot += s_cnt[q];
                if constexpr (TOMBS) again += s_reused[q];
            }
            int base = 0;
            if (tot > 0) {   // (who reuses a tombstone has a slot)
                base = again > 0 ? change_size(m.ctr, tot, -again) : atomicAdd(m.ctr + kCtrSize, tot);
                if (base + tot > m.capacity) {
                    const int lo = base > m.capacity ? base : m.capacity;
                    const int excess = base + tot - lo;
                    change_counter(m.ctr + kCtrSize, -excess);
                    change_counter(m.ctr + kCtrDropped, excess);
                }
            }
            s_base = base;
        }
        __syncthreads();
        int top = s_base + rank;
        for (int q = 0; q < wave; ++q) top += s_cnt[q];
        if (w) {
            if (top < m.capacity) {
                idx = m.heap[top];   // (addresses a row: check_heap_kernel)
            } else {
                // Heap exhausted: give the slot up again.
                if (won) {
                    atomicExch(slot_ptr(m, wb, ws), kTomb);
                } else {
                    __hip_atomic_store(m.gstate + gp, kGenTomb,
                                       __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                    change_counter(m.ctr + kCtrGenTombs, 1);
                }
                change_counter(m.ctr + kCtrTombs, 1);
            }
        }
    }
    if (idx >= 0) {
        // (0 <= idx < capacity: heap entries are, loaded indices were checked)
        if (won) {
            *value_ptr(m, wb, ws) = idx;
            m.klog[idx] = code;
        } else {
            __hip_atomic_store(m.gstate + gp, idx, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            m.klog[idx] = kTomb;   // "stored in the general region"
            change_counter(m.ctr + kCtrGenLive, 1);
        }
        if constexpr (MODE == kInsertFused) {
            // (four words at a time: word after word, each was waited for by its store)
#pragma unroll 1
            for (int v = 0; v < va.n; ++v) {
                const int rd = va.row_dwords[v];
                const uint32_t* s = va.src[v] + i * rd;
                uint32_t* d = va.dst[v] + static_cast<int64_t>(idx) * rd;
#pragma unroll 1
                for (int q = 0; q < rd; q += 4) {
                    uint32_t word[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) word[k] = q + k < rd ? s[q + k] : 0u;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        if (q + k < rd) d[q + k] = word[k];
                    }
                }
            }
        }
    }
    if constexpr (MODE == kInsertAssign) {
        if (active) assigned[i] = idx;
    }
    if constexpr (MODE == kInsertReport) {
        // The index of the key, if this thread can be sure of it: the one it
        // was given just now, or the one read beside a key that was there --
        // but a key that another thread is storing in this very launch shows
        // before its index is written, and the word beside it still holds
        // whatever an earlier tenant of the slot left.  The key log settles
        // it: klog[index] names this key only if that index is the key's own.
        // (-1 tells the caller that the thread storing the key will know.)
        int32_t r = idx;
        if (r < 0 && static_cast<uint32_t>(seen) < static_cast<uint32_t>(m.capacity) &&
            m.klog[seen] == code) {
            r = seen;
        }
        if (r < 0 && gdup) {
            // (the general region shows an index only once it is final)
            uint32_t at;
            int32_t gi;
            if (gen_find<DIM>(m, k, gi, at)) r = gi;
        }
        *report = r;
    }
}

// One key per thread, every thread of the workgroup calls this together.
// CODES: `keys` holds packed 64-bit codes instead of int32[DIM] rows.
template <int DIM, int MODE, bool TOMBS, bool CODES, int BLOCK = kHeapBlock, bool ALONE = false>
__device__ __forceinline__ void insert_one(
        const MapDev& m, const int32_t* __restrict__ keys, int64_t i,
        bool active, const ValueArgs& va, int32_t* __restrict__ assigned,
        const int64_t* __restrict__ given) {
    int32_t k[DIM] = {};
    uint64_t code;
    bool fits;
    if constexpr (CODES) {
        code = active ? reinterpret_cast<const uint64_t*>(keys)[i] : 0ull;
        fits = true;
    } else {
        load_key<DIM>(keys, i, active, k);
        fits = pack_key<DIM>(k, code);
    }
    insert_key<DIM, MODE, TOMBS, BLOCK, ALONE>(m, k, code, fits, i, active, va, assigned, given);
}

// The counters, left where the host reads them: `landing` is a place in page-locked
// host memory (kLineWords).  For one workgroup.  (Atomic reads: like every change
// of a counter they are made where all XCDs meet.)
__device__ __forceinline__ void leave_counters(const int32_t* ctr, uint64_t* landing, int32_t stamp) {
    if (threadIdx.x < kHostCounters) {
        leave_word(landing + threadIdx.x,
                   __hip_atomic_load(ctr + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), stamp);
    }
}

// The end of a launch that changes the counters: its last workgroup leaves them for
// the host (`publish`, where there is a landing place), which saves a launch behind
// it.  Every thread calls this, and has waited for the changes it has made
// (change_counter).  No fence: one per wavefront has the L2 written back each time
// (65 537 keys that take a few tombstones per workgroup: 18 -> 40 us, and erased
// again 12 -> 28; as it is 18 and 12).
// `groups`: the workgroups that come here.
__device__ __forceinline__ void leave_with_last(const MapDev& m, const Publish& publish,
                                                unsigned groups) {
    if (publish.landing == nullptr) return;
    __shared__ bool s_last;
    __syncthreads();
    if (threadIdx.x == 0) {
        s_last = atomicAdd(publish.ticket, 1) == static_cast<int32_t>(groups) - 1;
        if (s_last) atomicExch(publish.ticket, 0);
    }
    __syncthreads();
    if (s_last) leave_counters(m.ctr, publish.landing, publish.stamp);
}

// What the host waits for before it returns from an insert: whether every key fits the
// packed code.  (One that does not wants the second region attached, or may find that
// full while the table is not: the counters are read then.)  The first `groups` workgroups of
// the launch (none: nobody waits) look at all keys and at nothing else, and the last
// of them leaves the number of workgroups that have met one that does not fit.  That
// is there as soon as the launch has begun, and what follows the insert is queued
// while it runs; from its counters, behind it, the host knew only when it was done
// (a batch of 65 537 that comes, is read and goes: 101.5 us, 90 this way; a map of 1000
// keys filled and read back 45.5 -> 34).
struct KeyCheck {
    unsigned groups;
    uint64_t* word;    // page-locked
    int32_t stamp;
    int32_t* ticket;   // zero before and after
};
constexpr int kCheckKeys = 16;   // per thread: a few turns of four loads
constexpr unsigned kMostChecks = 256;

template <int DIM, int BLOCK>
__device__ __forceinline__ void check_keys(const int32_t* __restrict__ keys, int64_t n,
                                           const KeyCheck& check) {
    bool bad = false;
    const int64_t stride = static_cast<int64_t>(check.groups) * BLOCK;
#pragma unroll 4
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * BLOCK + threadIdx.x; i < n; i += stride) {
        int32_t k[DIM];
        load_key<DIM>(keys, i, true, k);
        uint64_t code;
        bad = bad | !pack_key<DIM>(k, code);
    }
    bad = __syncthreads_or(bad) != 0;
    if (threadIdx.x != 0) return;
    constexpr int kBad = 1 << 16;
    static_assert(kMostChecks < kBad, "workgroups below, those that met such a key above");
    const int32_t before = atomicAdd(check.ticket, bad ? kBad + 1 : 1);
    if ((before & (kBad - 1)) != static_cast<int32_t>(check.groups) - 1) return;
    atomicExch(check.ticket, 0);
    leave_word(check.word, (before >> 16) + (bad ? 1 : 0), check.stamp);
}

template <int DIM, int MODE, bool TOMBS, int BLOCK, bool ALONE>
__global__ __launch_bounds__(BLOCK) void insert_kernel(
        MapDev m, const int32_t* __restrict__ keys, int64_t n, ValueArgs va,
        int32_t* __restrict__ assigned, const int64_t* __restrict__ given, Publish publish,
        KeyCheck check) {
    if (blockIdx.x < check.groups) return check_keys<DIM, BLOCK>(keys, n, check);
    const int64_t i = static_cast<int64_t>(blockIdx.x - check.groups) * BLOCK + threadIdx.x;
    insert_one<DIM, MODE, TOMBS, false, BLOCK, ALONE>(m, keys, i, i < n, va, assigned, given);
    leave_with_last(m, publish, gridDim.x - check.groups);
}

// The same insert over a selection made on the device: thread t of the
// selection handles row sel[t], t < *nsel.  The grid is fixed; workgroups
// stride over the selection, which is empty in the common case.
template <int DIM, int MODE, bool TOMBS, bool CODES>
__global__ __launch_bounds__(kHeapBlock) void insert_selected_kernel(
        MapDev m, const int32_t* __restrict__ keys,
        const int32_t* __restrict__ sel, const int32_t* __restrict__ nsel,
        ValueArgs va, Publish publish) {
    const int64_t total = *nsel;
    for (int64_t base = static_cast<int64_t>(blockIdx.x) * kHeapBlock;
         base < total; base += static_cast<int64_t>(gridDim.x) * kHeapBlock) {
        const int64_t t = base + threadIdx.x;
        const bool active = t < total;
        const int64_t i = active ? sel[t] : 0;
        insert_one<DIM, MODE, TOMBS, CODES>(m, keys, i, active, va, nullptr, nullptr);
        __syncthreads();
    }
    if (publish.landing == nullptr) return;
    if (total == 0) {   // nothing has changed the counters
        if (blockIdx.x != 0) return;
    } else {            // the workgroup that ends last
        __shared__ bool s_last;
        __threadfence();
        __syncthreads();
        if (threadIdx.x == 0) s_last = atomicAdd(publish.ticket, 1) == static_cast<int32_t>(gridDim.x) - 1;
        __syncthreads();
        if (!s_last) return;
    }
    leave_counters(m.ctr, publish.landing, publish.stamp);
}

// Block activation around a batch of positions (ash/grid.py:121-159): the
// block of every position and its neighbours within the dilation are inserted
// as int3 keys.  The reference expands every position into (2r+1)^3 candidate
// rows, de-duplicates them through a scratch hash set and inserts the
// survivors.  Here positions arrive in image order, so their blocks come in
// runs: activate_heads_kernel keeps one block per run ("head", one atomic per
// wavefront to reserve list space), and activate_kernel then handles one
// (head, neighbour offset) pair per thread, the table absorbing the remaining
// duplicates.  MARK = false inserts; MARK = true (a second launch, when every
// index is final) looks the candidates up again, flags their rows in `touched`
// and records their coordinates, from which the caller lists the touched
// blocks.
__device__ __forceinline__ bool block_of_position(
        const float* __restrict__ cells, int64_t i, float g, int bound_lo,
        int bound_hi, int32_t (&base)[3]) {
    bool inside = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        base[d] = static_cast<int32_t>(floorf(__fdiv_rn(cells[i * 3 + d], g)));
        inside = inside && base[d] >= bound_lo && base[d] <= bound_hi;
    }
    return inside;
}

// heads[0] = number of heads (zero on entry), heads[64 + 3 h ..] = block h.
// One update of the shared counter per 1024 positions.
constexpr int kHeadsBlock = 1024;

__global__ __launch_bounds__(kHeadsBlock) void activate_heads_kernel(
        const float* __restrict__ cells, int64_t n, float g, int bound_lo,
        int bound_hi, int32_t* __restrict__ heads) {
    __shared__ int s_cnt[kHeadsBlock / 64];
    __shared__ int s_first;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kHeadsBlock + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    int32_t base[3] = {0, 0, 0};
    bool lead = false;
    if (i < n) {
        lead = block_of_position(cells, i, g, bound_lo, bound_hi, base);
        if (lead && i > 0) {
            int32_t prev[3];
            const bool pin = block_of_position(cells, i - 1, g, bound_lo, bound_hi, prev);
            lead = !pin || prev[0] != base[0] || prev[1] != base[1] || prev[2] != base[2];
        }
    }
    const uint64_t lm = __ballot(lead);
    if (lane == 0) s_cnt[wave] = __popcll(lm);
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
#pragma unroll
        for (int q = 0; q < kHeadsBlock / 64; ++q) {
            const int c = s_cnt[q];
            s_cnt[q] = tot;
            tot += c;
        }
        s_first = tot ? atomicAdd(heads, tot) : 0;
    }
    __syncthreads();
    if (lead) {
        int32_t* out = heads + 64 +
                       3 * static_cast<int64_t>(s_first + s_cnt[wave] +
                                                __popcll(lm & ((1ull << lane) - 1ull)));
        out[0] = base[0];
        out[1] = base[1];
        out[2] = base[2];
    }
}

template <bool MARK, bool TOMBS>
__global__ __launch_bounds__(kHeapBlock) void activate_kernel(
        MapDev m, const int32_t* __restrict__ heads, int off_lo, int width,
        int bound_lo, int bound_hi, uint8_t* __restrict__ touched,
        int32_t* __restrict__ coords) {
    const int per_head = width * width * width;
    const int64_t total = static_cast<int64_t>(heads[0]) * per_head;
    const ValueArgs none = {};
    for (int64_t first = static_cast<int64_t>(blockIdx.x) * kHeapBlock; first < total;
         first += static_cast<int64_t>(gridDim.x) * kHeapBlock) {
        const int64_t t = first + threadIdx.x;
        bool ok = t < total;
        int32_t k[3] = {0, 0, 0};
        if (ok) {
            const int64_t h = t / per_head;
            const int o = static_cast<int>(t - h * per_head);
            const int32_t* base = heads + 64 + 3 * h;
            k[0] = base[0] + off_lo + o % width;
            k[1] = base[1] + off_lo + (o / width) % width;
            k[2] = base[2] + off_lo + o / (width * width);
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                ok = ok && k[d] >= bound_lo && k[d] <= bound_hi;
            }
        }
        if constexpr (!MARK) {
            uint64_t code;
            const bool fits = pack_key<3>(k, code);
            insert_key<3, kInsertKeys, TOMBS>(m, k, code, fits, 0, ok, none, nullptr, nullptr);
            __syncthreads();
        } else {
            int32_t idx = 0;
            const bool found = find_key<3>(m, k, ok, idx);
            if (found && ok) {
                touched[idx] = 1;
                coords[static_cast<int64_t>(idx) * 3 + 0] = k[0];
                coords[static_cast<int64_t>(idx) * 3 + 1] = k[1];
                coords[static_cast<int64_t>(idx) * 3 + 2] = k[2];
            }
        }
    }
}

// The same activation straight from world positions, without a list of run
// heads in memory: a workgroup finds the heads among its own kRunPositions
// positions (a position leads a run when the position before it lies in
// another block, whichever workgroup that one belongs to), keeps them in LDS
// and handles their (head, neighbour offset) pairs itself: no list to write
// and read back, no counter to clear.
// Positions are in world units: cell units = (x - origin) * inv_cell, evaluated
// as torch evaluates `(x - origin) / cell_size` on the device (grid_forward's
// front end does the same); origin null and inv_cell 1 leave them as they are.
struct RunsArgs {
    const float* x;        // float32[n, 3]
    const float* origin;   // float32[3] on the device, or nullptr
    float inv_cell;
    float g;               // cells per block edge
    int64_t n;
    int off_lo, width;     // neighbour offsets off_lo .. off_lo + width - 1 per axis
    int bound_lo, bound_hi;
    bool empty;            // the table holds nothing yet
};

__device__ __forceinline__ bool block_of_world(const RunsArgs& a, int64_t i,
                                               int32_t (&base)[3]) {
    bool inside = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float o = a.origin != nullptr ? a.origin[d] : 0.f;
        const float c = __fmul_rn(__fsub_rn(a.x[i * 3 + d], o), a.inv_cell);
        base[d] = static_cast<int32_t>(floorf(__fdiv_rn(c, a.g)));
        inside = inside && base[d] >= a.bound_lo && base[d] <= a.bound_hi;
    }
    return inside;
}

constexpr int kRunPositions = 256;
static_assert(kRunPositions % 64 == 0 && kRunPositions <= kHeapBlock, "whole wavefronts of positions");
constexpr int kCandChunk = 1024;         // candidates made distinct at a time
constexpr int kDistinctSlots = 2048;     // two LDS slots per candidate of a chunk

// One launch per batch: insert and flag.  The (head, neighbour offset)
// candidates of a workgroup -- 570 for 256 pixels of a VGA frame at dilation 1 --
// name every block twice on average (the neighbourhoods of neighbouring
// blocks overlap in 18 of 27), so they are first made distinct in an LDS set,
// and then looked up by a lane each, one after the other without a barrier in
// between: a block that stands, which is what a frame mostly meets, is flagged there
// and then, once the key log confirms its index.  (A table that has been emptied and not
// used since holds none, and is not looked at.)  What is left is inserted.  The insert
// reports the index of every key it can be sure of (insert_key, kInsertReport)
// and the row is flagged at once; a key that another thread is storing at
// that moment is flagged by that thread, which is handed the index.  No second
// launch has to wait for the indices to settle.
//
// ALONE: the insert's lanes look at their buckets by themselves, with the index along with
// the codes, as other workgroups' atomics take the lines away.  Into emptied tables only
// up to two workgroups per CU: beyond, all of them meet in the same buckets at once, and
// the quicker probe makes more of their atomics fail (VGA frame 27.6 -> 30.2 us; 160 x
// 120 32.0 -> 27.2).
//
// A chain of waits.  Every block through a cooperative insert | that insert behind the look
// | as it is (us), by the share of a frame's blocks that are new to a standing table, at one
// side of it: VGA frame, 817 workgroups of some 250 distinct blocks, none 14.7 | 12.5 | 12.5,
// 3 % 17.4 | 18.0 | 16.0, 10 % 20.5 | 20.6 | 17.6, half 24.0 | 24.8 | 22.9, all 28.4 | 31.6 |
// 32.2; 160 x 120 26 | 18.7 | 18.6, 27.5 | 25.8 | 22.9, 28.4 | 27.2 | 24.1, 31 | 29.6 | 26.7,
// 33 | 37 | 33; 1200 x 900 25 | 21 | 21, 30 | 31 | 25, 38 | 39 | 29, 52 | 57 | 45, 63 | 68 |
// 62; VGA with blocks of twice the edge 10.2 | 8.3 | 8.8, 11.4 | 13.8 | 12.8, 15.1 | 15.7 |
// 15.1, 21 | 21 | 23, 26 | 28 | 30.  (Frames of which everything is new are better off without the
// look, which nobody knows beforehand.)  512 threads, one round for everybody: 16, the
// registers of the insert leave room for half of the workgroups; 128 and 64 positions 16.6
// and 23.
template <bool TOMBS, bool ALONE>
__global__ __launch_bounds__(kHeapBlock) void activate_runs_kernel(
        MapDev m, RunsArgs a, uint8_t* __restrict__ touched, int32_t* __restrict__ coords) {
    __shared__ unsigned long long s_set[kDistinctSlots];
    __shared__ int32_t s_cand[kCandChunk * 3];
    __shared__ int32_t s_heads[kRunPositions * 3];
    __shared__ int s_wave[kRunPositions / 64];
    __shared__ int s_ncand;
    __shared__ int s_nmissing;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kRunPositions + threadIdx.x;
    int32_t base[3] = {0, 0, 0};
    bool lead = false;
    if (threadIdx.x < kRunPositions && i < a.n) {
        lead = block_of_world(a, i, base);
        if (lead && i > 0) {
            int32_t prev[3];
            const bool pin = block_of_world(a, i - 1, prev);
            lead = !pin || prev[0] != base[0] || prev[1] != base[1] || prev[2] != base[2];
        }
    }
    const uint64_t lm = __ballot(lead);
    if (lane == 0 && wave < kRunPositions / 64) s_wave[wave] = __popcll(lm);
    __syncthreads();
    int before = 0, nh = 0;
#pragma unroll
    for (int q = 0; q < kRunPositions / 64; ++q) {
        const int c = s_wave[q];
        if (q < wave) before += c;
        nh += c;
    }
    if (lead) {
        const int h = before + __popcll(lm & ((1ull << lane) - 1ull));
        s_heads[h * 3 + 0] = base[0];
        s_heads[h * 3 + 1] = base[1];
        s_heads[h * 3 + 2] = base[2];
    }
    const int per_head = a.width * a.width * a.width;
    const int total = nh * per_head;   // the same for every thread of the workgroup
    const ValueArgs none = {};
    auto flag = [&](int32_t row, const int32_t (&k)[3]) {
        touched[row] = 1;
        coords[static_cast<int64_t>(row) * 3 + 0] = k[0];
        coords[static_cast<int64_t>(row) * 3 + 1] = k[1];
        coords[static_cast<int64_t>(row) * 3 + 2] = k[2];
    };
    for (int first = 0; first < total; first += kCandChunk) {
        for (int q = threadIdx.x; q < kDistinctSlots; q += kHeapBlock) s_set[q] = kEmpty;
        if (threadIdx.x == 0) s_ncand = s_nmissing = 0;
        __syncthreads();   // (also: s_heads is complete, the rounds below are over)
        const int end = total - first < kCandChunk ? total : first + kCandChunk;
        for (int t = first + threadIdx.x; t < end; t += kHeapBlock) {
            const int h = t / per_head;
            const int o = t - h * per_head;
            int32_t c[3];
            c[0] = s_heads[h * 3 + 0] + a.off_lo + o % a.width;
            c[1] = s_heads[h * 3 + 1] + a.off_lo + (o / a.width) % a.width;
            c[2] = s_heads[h * 3 + 2] + a.off_lo + o / (a.width * a.width);
            bool keep = true;
#pragma unroll
            for (int d = 0; d < 3; ++d) keep = keep && c[d] >= a.bound_lo && c[d] <= a.bound_hi;
            uint64_t code;
            if (keep && pack_key<3>(c, code)) {   // (keys that do not pack are all kept)
                uint32_t at = static_cast<uint32_t>(mix64(code)) & (kDistinctSlots - 1);
                for (;;) {   // at most half of the slots are ever taken
                    const unsigned long long old = atomicCAS(&s_set[at], kEmpty, code);
                    if (old == kEmpty) break;
                    if (old == code) {
                        keep = false;
                        break;
                    }
                    at = (at + 1) & (kDistinctSlots - 1);
                }
            }
            if (keep) {
                const int at = atomicAdd(&s_ncand, 1);
                s_cand[at * 3 + 0] = c[0];
                s_cand[at * 3 + 1] = c[1];
                s_cand[at * 3 + 2] = c[2];
            }
        }
        __syncthreads();
        const int distinct = s_ncand;
        // blocks that stand, and whose index is certain, are flagged by whoever looks
        // them up; the others, none as a rule, are listed (over the set, which is done with)
        int32_t* const s_missing = reinterpret_cast<int32_t*>(s_set);
        for (int t = threadIdx.x; t < (a.empty ? 0 : distinct); t += kHeapBlock) {
            const int32_t k[3] = {s_cand[t * 3 + 0], s_cand[t * 3 + 1], s_cand[t * 3 + 2]};
            uint64_t code;
            const bool fits = pack_key<3>(k, code);
            int32_t row = -1;
            bool stands = find_key_alone<3>(m, k, true, row);
            if (stands && fits) {
                stands = static_cast<uint32_t>(row) < static_cast<uint32_t>(m.capacity) && m.klog[row] == code;
            }
            if (stands) {
                flag(row, k);
            } else {
                s_missing[atomicAdd(&s_nmissing, 1)] = t;
            }
        }
        __syncthreads();
        const int missing = a.empty ? distinct : s_nmissing;
        for (int r0 = 0; r0 < missing; r0 += kHeapBlock) {
            const bool ok = r0 + static_cast<int>(threadIdx.x) < missing;
            int32_t k[3] = {0, 0, 0};
            if (ok) {
                const int t = a.empty ? r0 + static_cast<int>(threadIdx.x) : s_missing[r0 + threadIdx.x];
                k[0] = s_cand[t * 3 + 0];
                k[1] = s_cand[t * 3 + 1];
                k[2] = s_cand[t * 3 + 2];
            }
            uint64_t code;
            const bool fits = pack_key<3>(k, code);
            int32_t row = -1;
            insert_key<3, kInsertReport, TOMBS, kHeapBlock, ALONE>(m, k, code, fits, 0, ok, none, nullptr, nullptr, &row);
            if (ok && row >= 0) flag(row, k);
            __syncthreads();   // insert_key's own words are rewritten by the next round
        }
    }
}

// Workgroup size of erase: the heap counter and the tombstone counter are each
// updated once per workgroup, and updates of one address serialise (about 7 ns
// each), so larger groups pay off here: measured on 16 M stored keys,
// 256 threads with a tombstone update per wavefront 3.0 ms, 1024 threads with
// one update of each counter per workgroup 0.85 ms.
// Fewer keys are better spread over the CUs.  Lanes look at their buckets by themselves,
// as inserts do, but take the index along with the codes
// (probe_alone).  Cooperative with 1024 threads -> alone with the index read behind the
// codes -> as it is (us), stored keys beside 100 000 | four million: 16 000 9.1 -> 6.8 ->
// 6.3 | 11.1 -> 7.5 -> 7.3, 65 537 10.0 -> 11.0 -> 9.6 | 12.4 -> 10.8 -> 10.0, 98 000 11.5
// -> 12.9 -> 11.4 | 13.9 -> 12.6 -> 11.9, 131 000 13.6 -> 15.7 -> 13.3 | 16.1 -> 15.2 ->
// 13.7, 164 000 15.0 -> 18.2 -> 14.0 | 17.7 -> 17.2 -> 14.4, 400 000 42 -> 32 -> 27 | 33 ->
// 28 -> 26, 1.6 million 92 -> 92 -> 85 | 88 -> 96 -> 84, 3.1 million 175 -> 228 -> 178
// beside four; each key four times 131 000 13.7 -> 16.6 -> 13.0, 3.1 million 109 -> 126 -> 90;
// absent keys 131 000 7.1 -> 5.8 -> 6.5, 3.1 million 77 -> 62 -> 63.  Larger batches,
// cooperative -> as it is: stored keys, four million beside four 225 -> 205, eight beside
// sixteen 400 -> 378, sixteen beside sixteen 843 -> 772; absent ones 120 -> 125, 265 -> 225,
// 632 -> 426; each four times, four million 116 -> 108, each sixteen times, eight 248 -> 188.
// With 256 | 512 | 1024
// threads: 50 000 8.6 | 8.5 | 11.0, 98 000 12.9 | 11.3 | 11.9, 115 000 15.0 | 12.5 | 12.6,
// 131 000 17.9 | 14.1 | 13.3.
constexpr int kEraseBlock = 1024;
constexpr int64_t kEraseBy256 = int64_t{3} << 14, kEraseBy512 = int64_t{7} << 14;

// One key per thread, every thread of the workgroup calls this together.
// CODES: `keys` holds packed 64-bit codes instead of int32[DIM] rows.
template <int DIM, bool CODES, int BLOCK = kEraseBlock, bool ALONE = false>
__device__ __forceinline__ void erase_one(const MapDev& m, const int32_t* __restrict__ keys,
                                          int64_t i, bool active) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    int32_t k[DIM] = {};
    uint64_t code;
    bool fits;
    if constexpr (CODES) {
        code = active ? reinterpret_cast<const uint64_t*>(keys)[i] : 0ull;
        fits = true;
    } else {
        load_key<DIM>(keys, i, active, k);
        fits = pack_key<DIM>(k, code);
    }
    bool pend = active && fits;
    uint32_t b = bucket_of(code, m.nb);
    uint32_t steps = 0;
    bool won = false;
    bool tomb = false;
    int32_t idx = 0;
    while (__ballot(pend)) {
        ProbeResult p;
        if constexpr (ALONE) probe_alone(m, code, b, pend, p);
        else probe_pass(m, code, b, pend, lane, p);
        if (pend) {
            if (p.status == kProbeFound) {
                // A bucket that still has an empty slot has never been full,
                // so no key was ever pushed past it: the slot can go straight
                // back to empty.  Otherwise leave a tombstone.
                const bool reuse = p.emask != 0;
                const unsigned long long old = atomicCAS(
                        slot_ptr(m, b, p.slot), code, reuse ? kEmpty : kTomb);
                if (old == code) {
                    won = true;
                    tomb = !reuse;
                    idx = p.val;
                }
                pend = false;
            } else if (p.status == kProbeHasEmpty) {
                pend = false;
            } else {
                b = next_bucket(b, m.nb);
                if (++steps >= kPartBuckets) pend = false;
            }
        }
    }
    if (active && !fits) {
        int32_t gi;
        uint32_t pos;
        if (gen_find<DIM>(m, k, gi, pos)) {
            if (atomicCAS(m.gstate + pos, gi, kGenTomb) == gi) {
                won = true;
                tomb = true;
                idx = gi;
                change_counter(m.ctr + kCtrGenLive, -1);
                change_counter(m.ctr + kCtrGenTombs, 1);
            }
        }
    }
    __shared__ int s_cnt[BLOCK / 64];
    __shared__ int s_tomb[BLOCK / 64];
    __shared__ int s_base;
    const uint64_t wm = __ballot(won);
    const int nw = __popcll(wm);
    const int rank = __popcll(wm & ((1ull << lane) - 1ull));
    const int nt = __popcll(__ballot(tomb));
    if (lane == 0) {
        s_cnt[wave] = nw;
        s_tomb[wave] = nt;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0, tombs = 0;
#pragma unroll
        for (int q = 0; q < BLOCK / 64; ++q) {
            tot += s_cnt[q];
            tombs += s_tomb[q];
        }
        // (every tombstone is an entry that went)
        s_base = tombs > 0 ? change_size(m.ctr, -tot, tombs) : tot > 0 ? atomicSub(m.ctr + kCtrSize, tot) : 0;
    }
    __syncthreads();
    if (won) {
        int below = rank;
        for (int q = 0; q < wave; ++q) below += s_cnt[q];
        const int pos = s_base - 1 - below;
        if (pos >= 0 && pos < m.capacity) m.heap[pos] = idx;
        if (static_cast<uint32_t>(idx) < static_cast<uint32_t>(m.capacity)) m.klog[idx] = kEmpty;
    }
}

template <int DIM, int BLOCK>
__global__ __launch_bounds__(BLOCK) void erase_kernel(
        MapDev m, const int32_t* __restrict__ keys, int64_t n, Publish publish) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * BLOCK + threadIdx.x;
    erase_one<DIM, false, BLOCK, true>(m, keys, i, i < n);
    leave_with_last(m, publish, gridDim.x);
}

// The same erase over a selection made on the device (see
// insert_selected_kernel): thread t handles key sel[t], t < *nsel.
template <int DIM, bool CODES>
__global__ __launch_bounds__(kEraseBlock) void erase_selected_kernel(
        MapDev m, const int32_t* __restrict__ keys, const int32_t* __restrict__ sel,
        const int32_t* __restrict__ nsel) {
    const int64_t total = *nsel;
    for (int64_t base = static_cast<int64_t>(blockIdx.x) * kEraseBlock; base < total;
         base += static_cast<int64_t>(gridDim.x) * kEraseBlock) {
        const int64_t t = base + threadIdx.x;
        const bool active = t < total;
        erase_one<DIM, CODES>(m, keys, active ? sel[t] : 0, active);
        __syncthreads();   // the counters in LDS are free again
    }
}

// Rows of up to kMaxFusedValues tables, and where they are to go.
struct GatherArgs {
    int n;
    const uint32_t* src[kMaxFusedValues];
    uint32_t* dst[kMaxFusedValues];
    int32_t row_dwords[kMaxFusedValues];
    int64_t src_rows[kMaxFusedValues];
};

// items(): the live entries are read from the key log (8 bytes per index,
// against 21 bytes per index of bucket array).  A workgroup takes 1024 * ROUNDS
// consecutive indices, each of its wavefronts 64 * ROUNDS of them in rounds of
// 64, so that reads are contiguous and -- positions being ranks in index order
// -- so are the writes of every round; the entries of a workgroup come out
// sorted by index, workgroups in the order in which they reserve their output
// range.  `limit` indices are scanned: the capacity, or -- when nothing has
// written to the heap since it was last 0, 1, 2, ... (`identity`) and the
// indices in use therefore are 0 .. size-1 -- only the size.
// Output ranges come from one global cursor; atomics on that single address
// serialise (about 7 ns each across the XCDs), hence the large workgroups, of which
// there are as many as there are CUs while the table is small (items_rounds).  The
// upper half of the cursor counts the workgroups: the last sets it back to zero for
// the next listing, which a launch in front did before (`last`: nothing else goes on
// with the cursor).
// The value rows of an entry are copied along (`rows`: row_dwords words each): both
// sides run in index order.  Bound by memory from a million entries on (8 + 2 times
// the row bytes per index: 16 M in 24 M with rows of 16 bytes 287 -> 235 us, 5 TB/s),
// by the chain of accesses below; the rows by a launch of their own, which read the
// listed indices again, and the cursor's reset took two launches more (1.07 M in 1.6 M
// 25.2 -> 18.6, 67 000 in 100 000 11.3 -> 6.2).
constexpr int kItemsBlock = 1024;
constexpr int kItemsWaves = kItemsBlock / 64;

// items() while the heap is in its initial order and no key lives in the
// second region: the indices in use are 0 .. n-1, every one of them, so entry
// i of the output is index i and its key comes from log entry i -- no ranks,
// no cursor, and the value rows of the listed entries are the first n rows of
// every value tensor.
template <int DIM>
__global__ __launch_bounds__(kBlock) void items_dense_kernel(
        MapDev m, int32_t* __restrict__ keys_out, int64_t* __restrict__ idx_out, int64_t n) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    int32_t k[DIM];
    unpack_key<DIM>(m.klog[i], k);
#pragma unroll
    for (int d = 0; d < DIM; ++d) keys_out[i * DIM + d] = k[d];
    idx_out[i] = i;
}

template <int DIM, int ROUNDS>
__global__ __launch_bounds__(kItemsBlock) void items_kernel(
        MapDev m, int32_t* __restrict__ keys_out, int64_t* __restrict__ idx_out,
        int64_t n_expected, int identity, GatherArgs rows, int slot, bool last) {
    constexpr int kCounts = kItemsWaves * ROUNDS;
    static_assert(kCounts <= 128, "two wavefronts add them up");
    __shared__ int s_cnt[kCounts];
    __shared__ int s_base;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    unsigned long long* cursor = reinterpret_cast<unsigned long long*>(m.ctr + kCtrCursors) + slot;
    constexpr unsigned long long kDone = 1ull << 32;
    const unsigned long long all_but_one = (gridDim.x - 1ull) << 32;
    const int64_t limit = identity ? static_cast<int64_t>(m.ctr[kCtrSize])
                                   : static_cast<int64_t>(m.capacity);
    const int64_t first = static_cast<int64_t>(blockIdx.x) * (kItemsBlock * ROUNDS);
    const int64_t mine = first + wave * (64 * ROUNDS) + lane;
    uint64_t code[ROUNDS];
    int rank[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const int64_t i = mine + r * 64;
        code[r] = i < limit ? m.klog[i] : kEmpty;
    }
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const uint64_t live = __ballot(code[r] < kTomb);
        rank[r] = __popcll(live & ((1ull << lane) - 1ull));
        if (lane == 0) s_cnt[wave * ROUNDS + r] = __popcll(live);
    }
    __syncthreads();
    // exclusive scan of the counts by the first two wavefronts
    const bool scanner = threadIdx.x < kCounts;
    int c = 0, incl = 0;
    if (scanner) {
        c = s_cnt[threadIdx.x];
        incl = c;
    }
    if (threadIdx.x < 128) {
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int up = __shfl_up(incl, d);
            if (lane >= d) incl += up;
        }
    }
    __syncthreads();
    if (scanner) {
        s_cnt[threadIdx.x] = incl - c;
        if (threadIdx.x == 63) s_base = incl;   // total of the first 64 counts
    }
    __syncthreads();
    if (scanner && threadIdx.x >= 64) s_cnt[threadIdx.x] += s_base;
    __syncthreads();
    if (threadIdx.x == kCounts - 1) {
        const unsigned long long at =
                atomicAdd(cursor, kDone + static_cast<unsigned long long>(s_cnt[threadIdx.x] + c));
        s_base = static_cast<int>(static_cast<uint32_t>(at));
        // (everybody else has been here)
        if (last && (at & ~(kDone - 1)) == all_but_one) atomicExch(cursor, 0ull);
    }
    __syncthreads();
    uint64_t live[ROUNDS];   // of the 64 entries of a round, and where the first goes
    int64_t to[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        live[r] = __ballot(code[r] < kTomb);
        to[r] = static_cast<int64_t>(s_base) + s_cnt[wave * ROUNDS + r];
        const int64_t pos = to[r] + rank[r];
        if (code[r] < kTomb && pos < n_expected) {
            int32_t k[DIM];
            unpack_key<DIM>(code[r], k);
#pragma unroll
            for (int d = 0; d < DIM; ++d) keys_out[pos * DIM + d] = k[d];
            idx_out[pos] = mine + r * 64;
        }
    }
    // The rows of a round's 64 indices are one stretch of the source; lanes walk along
    // it, so that both sides are read and written whole (a lane per row and word after
    // word: 4 M entries with rows of 16 bytes 80 -> 54 us).
    for (int v = 0; v < rows.n; ++v) {
        const uint32_t rd = static_cast<uint32_t>(rows.row_dwords[v]);
        const uint32_t magic = 0xFFFFFFFFu / rd + 1u;   // (t / rd below 64 * rd, rd > 1)
        const uint32_t* __restrict__ src = rows.src[v] + (mine - lane) * rd;
        uint32_t* __restrict__ dst = rows.dst[v];
        const int64_t have = rows.src_rows[v] - (mine - lane);   // beyond it rows read as zeros
        for (uint32_t t = lane; t < 64u * rd; t += 64u) {
            const uint32_t row = rd == 1u ? t : __umulhi(t, magic);
            const uint64_t before = (1ull << row) - 1ull;
            uint32_t w[ROUNDS];
#pragma unroll
            for (int r = 0; r < ROUNDS; ++r) {
                const bool in = ((live[r] >> row) & 1ull) && row + r * 64 < have;
                w[r] = in ? src[static_cast<int64_t>(r) * 64 * rd + t] : 0u;
            }
#pragma unroll
            for (int r = 0; r < ROUNDS; ++r) {
                const int64_t pos = to[r] + __popcll(live[r] & before);
                if (((live[r] >> row) & 1ull) && pos < n_expected) dst[pos * rd + (t - row * rd)] = w[r];
            }
        }
    }
}

template <int DIM>
__global__ __launch_bounds__(kBlock) void items_general_kernel(
        MapDev m, int32_t* __restrict__ keys_out, int64_t* __restrict__ idx_out,
        int64_t n_expected, int32_t* __restrict__ cursor) {
    const uint32_t p = blockIdx.x * kBlock + threadIdx.x;
    const int lane = threadIdx.x & 63;
    int32_t w = kGenEmpty;
    if (p < m.gslots) w = m.gstate[p];
    const bool live = w >= 0;
    const uint64_t lm = __ballot(live);
    if (lm == 0) return;
    const int rank = __popcll(lm & ((1ull << lane) - 1ull));
    int base = 0;
    if (lane == 0) base = atomicAdd(cursor, __popcll(lm));
    base = __shfl(base, 0);
    if (live) {
        const int64_t pos = static_cast<int64_t>(base) + rank;
        if (pos < n_expected) {
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                keys_out[pos * DIM + d] = m.gkeys[static_cast<size_t>(p) * 4 + d];
            }
            idx_out[pos] = w;
        }
    }
}

// The neighbour table of every row (one launch instead of a listing, a batch of
// keys, their find and the scattering of both): a lane per row and offset, the
// row's key from the log, `width`^3 offsets with the first axis fastest, each
// `pad` less than its digit.  Rows without a key and offsets without a stored
// neighbour get -1.  A lane looks its neighbour up by itself, and the widths of the
// functions here are constants of their own: bound by vector instructions, of which the
// cooperative probe and divisions by a width from memory were the most (752 of a wavefront;
// 60 000 blocks of a surface, 8 offsets 15.3 -> 9.1 us (11 where other work has taken the
// caches in between), 27 offsets 34.7 -> 23.8; 200 000
// blocks 37 -> 25 and 106 -> 80; a million scattered ones, lines from behind the L2s, 197
// -> 123 and 657 -> 431; by a listing, a find and the scattering of both 80 us for the first).
struct NeighborArgs {
    int32_t* coords;   // [rows, 3]
    int64_t* lut;      // [rows, width^3]
    int64_t rows;
    int width, pad;
};

// every lane of the wavefront calls this together; lane `k` of row i.  WIDTH: the
// width, where it is not 0.
template <int WIDTH>
__device__ __forceinline__ void write_neighbor(const MapDev& m, const NeighborArgs& a, bool write,
                                               bool live, int64_t i, uint32_t k, const int32_t (&key)[3]) {
    const uint32_t w = static_cast<uint32_t>(WIDTH > 0 ? WIDTH : a.width);
    const uint32_t digit[3] = {k % w, k / w % w, k / w / w};
    int32_t other[3];
    bool self = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int32_t o = static_cast<int32_t>(digit[d]) - a.pad;
        self = self && o == 0;
        other[d] = static_cast<int32_t>(static_cast<uint32_t>(key[d]) + static_cast<uint32_t>(o));
    }
    int32_t res = 0;
    const bool found = find_key_alone<3>(m, other, live && !self, res);
    if (!write) return;
    a.lut[i * (w * w * w) + k] = live && self ? i : (found ? static_cast<int64_t>(res) : -1);
    if (k == 0) {
#pragma unroll
        for (int d = 0; d < 3; ++d) a.coords[i * 3 + d] = live ? key[d] : -1;
    }
}

// Share `block` of a workgroup: kBlock consecutive (row, offset) pairs.
template <int WIDTH>
__device__ __forceinline__ void row_and_offset(const NeighborArgs& a, int64_t block, int64_t& i,
                                               uint32_t& k) {
    const int w = WIDTH > 0 ? WIDTH : a.width;
    const uint32_t n = static_cast<uint32_t>(w * w * w);
    const int64_t base = block * kBlock;
    const uint32_t local = static_cast<uint32_t>(base % n) + threadIdx.x;
    i = base / n + local / n;
    k = local % n;
}

template <int WIDTH>
__global__ __launch_bounds__(kBlock) void neighbors_kernel(MapDev m, NeighborArgs a, int identity) {
    const int64_t limit = identity ? static_cast<int64_t>(m.ctr[kCtrSize])
                                   : static_cast<int64_t>(m.capacity);
    int64_t i;
    uint32_t k;
    row_and_offset<WIDTH>(a, blockIdx.x, i, k);
    const uint64_t code = i < limit && i < a.rows ? m.klog[i] : kEmpty;
    const bool live = code < kTomb;
    int32_t key[3] = {0, 0, 0};
    if (live) unpack_key<3>(code, key);
    write_neighbor<WIDTH>(m, a, i < a.rows, live, i, k, key);
}

// The same for the keys of the general region, behind it.
__global__ __launch_bounds__(kBlock) void neighbors_general_kernel(MapDev m, NeighborArgs a) {
    const int64_t shares = (static_cast<int64_t>(m.gslots) * a.width * a.width * a.width + kBlock - 1) / kBlock;
    for (int64_t share = blockIdx.x; share < shares; share += gridDim.x) {
        int64_t p;
        uint32_t k;
        row_and_offset<0>(a, share, p, k);
        const int32_t i = p < m.gslots ? m.gstate[p] : kGenEmpty;
        const bool live = i >= 0 && i < a.rows;
        int32_t key[3] = {0, 0, 0};
        if (live) {
#pragma unroll
            for (int d = 0; d < 3; ++d) key[d] = m.gkeys[static_cast<size_t>(p) * 4 + d];
        }
        write_neighbor<0>(m, a, live, live, i, k, key);
    }
}

__global__ __launch_bounds__(kBlock) void fill16_kernel(uint4* __restrict__ p,
                                                        int64_t n16,
                                                        uint32_t word) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock;
    const uint4 v = make_uint4(word, word, word, word);
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
         i < n16; i += stride) {
        p[i] = v;
    }
}

// klog[0 .. limit) := free, limit = the capacity or (prefix_only) the size
// counter -- or, if larger, the index below which an earlier clear left its
// entries standing -- rounded up to whole 16-byte units.  The log's allocation is a
// multiple of 16 bytes plus slack (256-byte aligned workspace regions), so the
// last unit of an odd capacity is written whole.
__global__ __launch_bounds__(kBlock) void empty_log_kernel(
        uint4* __restrict__ log16, int64_t capacity, const int32_t* __restrict__ ctr,
        int prefix_only) {
    int64_t entries = capacity;
    if (prefix_only) {
        const int64_t size = ctr[kCtrSize], high = ctr[kCtrLogHigh];
        const int64_t used = size > high ? size : high;
        entries = used < capacity ? used : capacity;
    }
    const int64_t n16 = (entries + 1) / 2;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock;
    const uint4 v = make_uint4(~0u, ~0u, ~0u, ~0u);
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < n16;
         i += stride) {
        log16[i] = v;
    }
}

// klog[size .. kCtrLogHigh) := free (8-byte stores: an odd size shares its
// 16 bytes with an entry in use).
__global__ __launch_bounds__(kBlock) void empty_log_tail_kernel(
        uint64_t* __restrict__ klog, int64_t capacity, const int32_t* __restrict__ ctr) {
    const int64_t from = ctr[kCtrSize] < 0 ? 0 : ctr[kCtrSize];
    const int64_t high = ctr[kCtrLogHigh];
    const int64_t to = high < capacity ? high : capacity;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock;
    for (int64_t i = from + static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < to;
         i += stride) {
        klog[i] = kEmpty;
    }
}

// The counters of an emptied table.  (Words of launches under way, kCtrTickets, are
// zero at rest and left alone.)
__global__ __launch_bounds__(kBlock) void reset_heap_kernel(
        int32_t* __restrict__ heap, int64_t capacity, int32_t* __restrict__ ctr,
        int32_t size_value, bool write_heap) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (write_heap && i < capacity) heap[i] = static_cast<int32_t>(i);
    if (i < kCtrTickets) ctr[i] = i == kCtrSize ? size_value : 0;
}

// A clear in one launch: counters, and stretches of memory that are filled with one
// word (value rows with zeros, the bucket array, the second region's states and the
// key log with ones) or counted up (the heap).  A piece of 16 bytes per thread, so
// that workgroups handed out one after the other walk through memory in order (four
// pieces: 200 MB 26.5 -> 26.0 us, but 512 MB 76 -> 86, 1.64 GB 240 -> 270).  Bound by the stores of large stretches (tables of 288 and
// 96 MB, with the counters: two fills of torch's and a launch for the counters 36.6 +
// 13.9 + 4.7 -> 48 us, 8.0 TB/s), and by the launch itself for small ones, which is
// why it is one (a launch in a busy stream costs 4 us however little it does; a set of
// 5640 keys emptied, filled and asked 41.5 -> 34.2 us).
constexpr int kClearSpans = kMaxFusedValues + 4;

struct ClearSpan {
    uint4* p;
    int64_t n16;       // whole pieces
    uint32_t word;
    uint8_t tail;      // bytes behind them
    bool count;        // 0, 1, 2, ... instead of `word`
    uint32_t first;    // the stretch's first workgroup
};

struct ClearArgs {
    int n;
    ClearSpan span[kClearSpans];
};

enum { kCountersAsTheyAre = 0, kCountersReset = 1, kCountersFresh = 2 };

// `counters`: left alone, reset, or those of a table that has never been used.  The
// key log beyond the size is left as it is where `keep_log`; kCtrLogHigh then
// remembers how far it may hold entries (the size so far, or what an earlier call
// remembered).
__global__ __launch_bounds__(kBlock) void clear_kernel(ClearArgs a, int32_t* __restrict__ ctr,
                                                       int counters, bool keep_log) {
    if (blockIdx.x == 0 && counters != kCountersAsTheyAre && threadIdx.x < kNumCounters) {
        // (one wavefront: every lane has read before any lane writes)
        const int i = threadIdx.x;
        const int32_t size = ctr[kCtrSize], high = ctr[kCtrLogHigh];
        int32_t v = 0;
        if (i == kCtrLogHigh && keep_log && counters == kCountersReset) v = size > high ? size : high;
        if (counters == kCountersFresh || i < kCtrTickets) ctr[i] = v;
    }
    if (a.n == 0) return;
    int k = 0;
    while (k + 1 < a.n && blockIdx.x >= a.span[k + 1].first) ++k;
    const ClearSpan& span = a.span[k];
    const int64_t i = static_cast<int64_t>(blockIdx.x - span.first) * kBlock + threadIdx.x;
    if (i < span.n16) {
        const uint32_t w = static_cast<uint32_t>(4 * i);
        span.p[i] = span.count ? make_uint4(w, w + 1, w + 2, w + 3)
                               : make_uint4(span.word, span.word, span.word, span.word);
    } else if (i == span.n16) {
        uint8_t* rest = reinterpret_cast<uint8_t*>(span.p + i);
        for (int b = 0; b < span.tail; ++b) {
            rest[b] = static_cast<uint8_t>((span.count ? static_cast<uint32_t>(4 * i) + b / 4 : span.word) >>
                                           (8 * (b % 4)));
        }
    }
}

// Keys counted as waiting for the second region although it is attached (a
// graph captured before the attach still runs without it) cannot be issued
// again by anybody: they are counted with the refused keys.
__global__ void fold_waiting_keys_kernel(int32_t* ctr) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        ctr[kCtrDropped] += ctr[kCtrExotic];
        ctr[kCtrExotic] = 0;
    }
}

__global__ void publish_counters_kernel(const int32_t* __restrict__ ctr, uint64_t* landing,
                                        int32_t stamp) {
    leave_counters(ctr, landing, stamp);
}

__global__ void set_counter_kernel(int32_t* ctr, int which, int32_t value) {
    if (threadIdx.x == 0 && blockIdx.x == 0) ctr[which] = value;
}

template <typename Unit>
__global__ __launch_bounds__(kBlock) void scatter_rows_kernel(
        const Unit* __restrict__ src, Unit* __restrict__ dst,
        const int32_t* __restrict__ assigned, int64_t n, int64_t units_per_row) {
    const int64_t total = n * units_per_row;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock;
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
         t < total; t += stride) {
        const int64_t row = t / units_per_row;
        const int64_t u = t - row * units_per_row;
        const int32_t a = assigned[row];
        if (a >= 0) dst[static_cast<int64_t>(a) * units_per_row + u] = src[t];
    }
}

// Row gather for up to kMaxFusedValues tensors at once: word t of output plane
// v is word t % rd of row indices[t / rd] of source plane v.  One launch reads
// the indices once per word of a row (the repeats hit the first-level cache);
// with indices in ascending runs, as items() returns them, source reads are
// contiguous.  RD = row width in words, 0 = read it from the arguments.
template <int RD>
__device__ __forceinline__ void gather_plane(const uint32_t* __restrict__ src,
                                             uint32_t* __restrict__ dst, int rd_runtime,
                                             const int64_t* __restrict__ indices, int64_t n,
                                             int64_t src_rows) {
    const uint32_t rd = RD > 0 ? static_cast<uint32_t>(RD) : static_cast<uint32_t>(rd_runtime);
    const int64_t words = n * rd;
    const bool narrow = words <= 0xFFFFFFFFll;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock;
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; t < words;
         t += stride) {
        const int64_t row = narrow ? static_cast<int64_t>(static_cast<uint32_t>(t) / rd) : t / rd;
        const uint32_t q = static_cast<uint32_t>(t - row * rd);
        const int64_t from = indices[row];
        // an index outside the source reads as zero instead of faulting
        __builtin_nontemporal_store((from >= 0 && from < src_rows) ? src[from * rd + q] : 0u, dst + t);
    }
}

// The first n rows of every plane, copied: what the gather is while the listing
// has entry i under index i.  16 bytes per thread where both sides allow it;
// source and copy are each touched once (non-temporal hint).
__global__ __launch_bounds__(kBlock) void copy_first_rows_kernel(GatherArgs a, int64_t n) {
    typedef unsigned int v4u __attribute__((ext_vector_type(4)));
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock;
    const int64_t tid = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    for (int v = 0; v < a.n; ++v) {
        const uint32_t* __restrict__ src = a.src[v];
        uint32_t* __restrict__ dst = a.dst[v];
        const int64_t have = a.src_rows[v] < n ? a.src_rows[v] : n;   // rows beyond the source read as zero
        const int64_t words = n * a.row_dwords[v];
        const int64_t live = have * a.row_dwords[v];
        const bool wide = reinterpret_cast<uintptr_t>(src) % 16 == 0 &&
                          reinterpret_cast<uintptr_t>(dst) % 16 == 0;
        const int64_t quads = wide ? live / 4 : 0;
        for (int64_t t = tid; t < quads; t += stride) {
            __builtin_nontemporal_store(
                    __builtin_nontemporal_load(reinterpret_cast<const v4u*>(src) + t),
                    reinterpret_cast<v4u*>(dst) + t);
        }
        for (int64_t t = 4 * quads + tid; t < words; t += stride) dst[t] = t < live ? src[t] : 0u;
    }
}

__global__ __launch_bounds__(kBlock) void gather_rows_kernel(
        GatherArgs a, const int64_t* __restrict__ indices, int64_t n) {
    for (int v = 0; v < a.n; ++v) {
        switch (a.row_dwords[v]) {
            case 1:
                gather_plane<1>(a.src[v], a.dst[v], 1, indices, n, a.src_rows[v]);
                break;
            case 2:
                gather_plane<2>(a.src[v], a.dst[v], 2, indices, n, a.src_rows[v]);
                break;
            case 3:
                gather_plane<3>(a.src[v], a.dst[v], 3, indices, n, a.src_rows[v]);
                break;
            case 4:
                gather_plane<4>(a.src[v], a.dst[v], 4, indices, n, a.src_rows[v]);
                break;
            default:
                gather_plane<0>(a.src[v], a.dst[v], a.row_dwords[v], indices, n, a.src_rows[v]);
                break;
        }
    }
}

// ----------------------------------------------- look-up with rows, and back
// Row tables read by a look-up: row `index` of src[v] goes to row i of dst[v].
// Rows are units[v] pieces of 4 bytes, or of 16 where `wide` has bit v set
// (row size and both base addresses are multiples of 16).
struct RowTables {
    int n;
    uint32_t wide;
    const void* src[kMaxFusedValues];
    void* dst[kMaxFusedValues];
    uint32_t units[kMaxFusedValues];
    uint32_t magic[kMaxFusedValues];   // t / units == umulhi(t, magic) for t < 64 * units
    uint32_t src_rows[kMaxFusedValues];
};

// Longest row (in pieces) whose 64 * units numbers the multiplication above
// divides exactly: t * (magic * units - 2^32) < 64 * units * units < 2^32.
constexpr int64_t kMaxRowUnits = 8191;

// The rows of the 64 keys of a wavefront: `from` is the row lane L's key reads
// (negative: a row of zeros), `rows` how many of the 64 keys exist.  Lanes
// walk the output in order, so it is written whole and a row is read by
// neighbouring lanes; up to four pieces per lane are in flight.
template <typename Unit>
__device__ __forceinline__ void copy_found_rows(const Unit* __restrict__ src, Unit* __restrict__ dst,
                                                uint32_t units, uint32_t magic, uint32_t src_rows,
                                                int32_t from, int rows) {
    constexpr int kAhead = 4;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t total = static_cast<uint32_t>(rows) * units;
    for (uint32_t t0 = 0; t0 < total; t0 += 64 * kAhead) {
        Unit w[kAhead];
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
            const uint32_t t = t0 + a * 64 + lane;
            const uint32_t row = units == 1 ? t : __umulhi(t, magic);
            const int32_t at = __shfl(from, static_cast<int>(row & 63u));
            w[a] = Unit{};
            if (t < total && static_cast<uint32_t>(at) < src_rows) {
                w[a] = src[static_cast<size_t>(static_cast<uint32_t>(at)) * units + (t - row * units)];
            }
        }
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
            const uint32_t t = t0 + a * 64 + lane;
            if (t < total) __builtin_nontemporal_store(w[a], dst + t);
        }
    }
}

// ... and of all tables, for the wavefront's keys first .. first + 63 of n.
__device__ __forceinline__ void copy_rows_of_wave(const RowTables& tabs, int32_t from, int64_t first, int64_t n) {
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    if (first >= n) return;   // whole wavefronts leave together
    const int rows = n - first < 64 ? static_cast<int>(n - first) : 64;
    for (int v = 0; v < tabs.n; ++v) {
        const uint32_t units = tabs.units[v];
        const size_t at = static_cast<size_t>(first) * units;
        if ((tabs.wide >> v) & 1u) {
            copy_found_rows<u4>(static_cast<const u4*>(tabs.src[v]), static_cast<u4*>(tabs.dst[v]) + at,
                                units, tabs.magic[v], tabs.src_rows[v], from, rows);
        } else {
            copy_found_rows<uint32_t>(static_cast<const uint32_t*>(tabs.src[v]),
                                      static_cast<uint32_t*>(tabs.dst[v]) + at, units,
                                      tabs.magic[v], tabs.src_rows[v], from, rows);
        }
    }
}

// find and the gather of the rows in one launch: the indices never travel
// through memory unless the caller wants them, and the line of a key's bucket
// and the lines of its rows are asked for by the same wavefront.  16 M keys
// with rows of 12 and 4 bytes: see the table of the design notes.
template <int DIM, bool ALONE>
__global__ __launch_bounds__(kBlock) void find_rows_kernel(
        MapDev m, const int32_t* __restrict__ keys, int64_t n, RowTables tabs, int miss_row,
        int64_t* __restrict__ idx_out, uint8_t* __restrict__ mask_out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    const bool active = i < n;
    int32_t k[DIM];
    load_key<DIM>(keys, i, active, k);
    int32_t res = 0;
    const bool found = look_up<DIM, ALONE>(m, k, active, res);
    if (active) {
        if (idx_out != nullptr) idx_out[i] = found ? static_cast<int64_t>(res) : 0;
        if (mask_out != nullptr) mask_out[i] = found ? 1 : 0;
    }
    copy_rows_of_wave(tabs, found ? res : miss_row, i - (threadIdx.x & 63), n);
}

// ------------------------------------- look-up with rows, rows in index order
// find_rows_kernel asks for three random lines per key when two tables are read
// (bucket, row, row), and the device delivers 50 - 58 G random lines a second
// whatever part of a line is wanted and wherever behind the L2s it comes from (250
// G where an L2 has them): 16 M keys with rows of 12 and 4 bytes take 942 us, of
// which 600 are lines of rows.  Here the rows are read a part of the tables at a
// time, which then sits in an L2:
//   1. look-up; a chunk of kSortChunk queries is sorted by the part its indices
//      lie in (in LDS) and leaves its indices in that order, the bounds of its
//      parts and, for every query, its place in that order;
//   2. per part: the indices that all chunks have left for it, their rows copied
//      side by side to the indices' places (the workgroups of an XCD stand in
//      one or two parts at a time, see gather_parts_kernel);
//   3. per chunk: the rows, read through, dealt to the queries from LDS.
// A chunk with few stored keys gets its rows key by key in pass 1 (plan_row_sort).
// The look-up keeps its one random line per key; everything else streams: 2 + 4
// bytes per key out, 4 + row in, row out, 2 + row in.  Chunks own their regions, so
// there is nothing to count beforehand and nothing that can overflow, whatever the
// indices are.  The same 16 M keys: 359 (of them 300 for the buckets' lines) + 275
// + 99 us.  The second pass is bound by requests to the L2s, two per key; parts of
// 1/128 and 1/512 of the tables: 278 and 299 us, of 1/64, more than an L2 holds, 324.
constexpr int kSortThreads = 512;
constexpr int kSortKeys = 8;                            // per thread
constexpr int kSortChunk = kSortThreads * kSortKeys;
constexpr int kSortParts = 256;
static_assert(kSortParts % 8 == 0, "parts are dealt to eight XCDs");
constexpr int kSortBounds = kSortParts + 2;
// Records of a chunk and part that pass 2 takes; pass 3 reads the rows of further
// ones itself, so that a wavefront's work is bounded when queries crowd in few
// parts (8 M queries of one key: 719 us without the bound, 210 with it, 117 key by key)
constexpr uint32_t kSortLongest = 256;
constexpr int kSortMaxWords = 8;                        // of a query's rows, all tables together
constexpr int kSortRuns = 8;                            // chunks per wavefront of pass 2
constexpr int kSortAhead = 4;                           // groups of 64 records in flight there
constexpr uint32_t kNoPlace = 0xFFFFu;
// the last word of a chunk's bounds: a part of it is longer than kSortLongest; pass 1
// has written its rows
enum : uint16_t { kBoundsLong = 1, kBoundsServed = 2 };

struct RowSort {
    int64_t n;
    uint32_t chunks;
    uint32_t scale;       // part of index i: umulhi(i, scale)
    uint32_t words;       // of a query's rows
    int eighths;          // a chunk with fewer eighths of its keys stored is served key by key
    int32_t* index;       // chunks * kSortChunk, a chunk's in part order
    uint16_t* place;      // n
    uint16_t* bounds;     // chunks * kSortBounds: where a chunk's parts start, its end, kBounds*
    uint32_t* rows;       // chunks * kSortChunk * words
};

template <int DIM>
__global__ __launch_bounds__(kSortThreads) void find_sort_kernel(
        MapDev m, const int32_t* __restrict__ keys, RowSort sort, RowTables tabs, int miss_row,
        int64_t* __restrict__ idx_out, uint8_t* __restrict__ mask_out) {
    static_assert(kSortChunk <= 0xFFFF, "places and bounds are 16-bit words");
    __shared__ int32_t s_index[kSortChunk];
    __shared__ uint32_t s_where[kSortChunk];   // part << 16 | rank within the part
    __shared__ int32_t s_count[kSortParts];
    __shared__ int32_t s_first[kSortParts];
    __shared__ int32_t s_wave[kSortThreads / 64];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kSortChunk;
    static_assert(kSortParts <= kSortThreads, "a thread per part");
    if (tid < kSortParts) s_count[tid] = 0;
    __syncthreads();
    uint16_t* bounds = sort.bounds + static_cast<int64_t>(blockIdx.x) * kSortBounds;
#pragma unroll 1
    for (int j = 0; j < kSortKeys; ++j) {
        const int64_t i = base + j * kSortThreads + tid;
        const bool active = i < sort.n;
        int32_t k[DIM];
        load_key<DIM>(keys, i, active, k);
        int32_t res = 0;
        const bool found = find_key<DIM>(m, k, active, res);
        if (active) {
            if (idx_out != nullptr) idx_out[i] = found ? static_cast<int64_t>(res) : 0;
            if (mask_out != nullptr) mask_out[i] = found ? 1 : 0;
        }
        uint32_t where = ~0u;
        if (found) {
            // (an index beyond every table reads zeros in pass 2, in whichever part)
            uint32_t part = __umulhi(static_cast<uint32_t>(res), sort.scale);
            if (part >= kSortParts) part = kSortParts - 1;
            where = (part << 16) | static_cast<uint32_t>(atomicAdd(&s_count[part], 1));
        }
        s_index[j * kSortThreads + tid] = res;
        s_where[j * kSortThreads + tid] = where;
    }
    __syncthreads();
    const int count = tid < kSortParts ? s_count[tid] : 0;
    int incl = count;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int up = __shfl_up(incl, d);
        if (lane >= d) incl += up;
    }
    if (lane == 63) s_wave[tid >> 6] = incl;
    int32_t res[kSortKeys];
#pragma unroll
    for (int j = 0; j < kSortKeys; ++j) res[j] = s_index[j * kSortThreads + tid];
    __syncthreads();
    int first = incl - count, total = 0;
#pragma unroll
    for (int w = 0; w < kSortThreads / 64; ++w) {
        if (w < (tid >> 6)) first += s_wave[w];
        total += s_wave[w];
    }
    const int queries = sort.n - base < kSortChunk ? static_cast<int>(sort.n - base) : kSortChunk;
    if (total * 8 < sort.eighths * queries) {
        // the chunk's rows key by key; the other passes find nothing of it
        if (tid < kSortBounds) bounds[tid] = tid == kSortParts + 1 ? kBoundsServed : 0;
#pragma unroll 1
        for (int j = 0; j < kSortKeys; ++j) {
            const int q = j * kSortThreads + tid;
            copy_rows_of_wave(tabs, s_where[q] != ~0u ? s_index[q] : miss_row, base + (q & ~63), sort.n);
        }
        return;
    }
    if (tid < kSortParts) {
        s_first[tid] = first;
        bounds[tid] = static_cast<uint16_t>(first);
    }
    const int longer = __syncthreads_or(count > static_cast<int>(kSortLongest));
    if (tid == 0) {
        bounds[kSortParts] = static_cast<uint16_t>(total);
        bounds[kSortParts + 1] = longer ? kBoundsLong : 0;
    }
#pragma unroll
    for (int j = 0; j < kSortKeys; ++j) {
        const int64_t i = base + j * kSortThreads + tid;
        const uint32_t where = s_where[j * kSortThreads + tid];
        uint32_t place = kNoPlace;
        if (where != ~0u) {
            place = static_cast<uint32_t>(s_first[where >> 16]) + (where & 0xFFFFu);
            s_index[place] = (where & 0xFFFFu) < kSortLongest ? res[j] : ~res[j];
        }
        if (i < sort.n) sort.place[i] = static_cast<uint16_t>(place);
    }
    __syncthreads();
    for (int t = tid; t < total; t += kSortThreads) sort.index[base + t] = s_index[t];
}

// Pass 2: a wavefront copies the rows of one part for kSortRuns chunks (the first
// kSortLongest of a chunk's).  Workgroups are dealt to the XCDs in turn, so
// workgroup w serves the parts w mod 8 + 8 i, one after the other: what an XCD's
// workgroups stand in at a time is one or two parts, 1 / 256 of the tables each.  A
// lane copies one word of a row, always the same one, so that the words of a row are
// asked for together and the rows leave as whole lines.
template <int WORDS>
__global__ __launch_bounds__(kBlock) void gather_parts_kernel(RowTables tabs, RowSort sort,
                                                              uint32_t groups) {
    constexpr uint32_t kWaves = kBlock / 64;
    constexpr uint32_t kXcdCount = 8;
    constexpr int kRecords = 64 / WORDS;                              // per step
    constexpr int kSteps = (64 + kRecords - 1) / kRecords;            // for the records of 64 lanes
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t turn = blockIdx.x / kXcdCount;
    const uint32_t part = turn / groups * kXcdCount + blockIdx.x % kXcdCount;
    const uint32_t c0 = (turn % groups * kWaves + threadIdx.x / 64) * kSortRuns;
    if (c0 >= sort.chunks) return;   // whole wavefronts
    // lane r < kSortRuns: the run of chunk c0 + r
    uint32_t from = 0, count = 0;
    if (lane < kSortRuns && c0 + lane < sort.chunks) {
        const uint16_t* b = sort.bounds + static_cast<int64_t>(c0 + lane) * kSortBounds + part;
        from = b[0];
        count = b[1] - from;
        if (count > kSortLongest) count = kSortLongest;
    }
    uint32_t ends = count;
#pragma unroll
    for (int d = 1; d < kSortRuns; d <<= 1) {
        const uint32_t up = __shfl_up(ends, d);
        if (lane >= static_cast<uint32_t>(d)) ends += up;
    }
    // place of record t of run r: t + shift of r (modulo 2^32)
    const uint32_t shift = (c0 + lane) * kSortChunk + from - (ends - count);
    const uint32_t total = __shfl(ends, kSortRuns - 1);
    if (total == 0) return;
    // the lane's word: of which table, and where in its rows
    const uint32_t record = lane / WORDS, word = lane % WORDS;
    const uint32_t* column = nullptr;
    uint32_t units = 0, rows = 0, before = 0;
    for (int v = 0; v < tabs.n; ++v) {
        if (word >= before) {
            column = static_cast<const uint32_t*>(tabs.src[v]) + (word - before);
            units = tabs.units[v];
            rows = tabs.src_rows[v];
        }
        before += tabs.units[v];
    }
    for (uint32_t t0 = 0; t0 < total; t0 += 64 * kSortAhead) {
        uint32_t at[kSortAhead], index[kSortAhead];
#pragma unroll
        for (int a = 0; a < kSortAhead; ++a) {
            const uint32_t t = t0 + a * 64 + lane;
            uint32_t run = 0;
#pragma unroll
            for (int r = 0; r < kSortRuns - 1; ++r) {
                run += t >= static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(ends), r)) ? 1u : 0u;
            }
            at[a] = t + static_cast<uint32_t>(__shfl(static_cast<int>(shift), static_cast<int>(run)));
            index[a] = t < total ? static_cast<uint32_t>(sort.index[at[a]]) : 0u;
        }
        uint32_t w[kSortAhead][kSteps];
#pragma unroll
        for (int a = 0; a < kSortAhead; ++a) {
#pragma unroll
            for (int st = 0; st < kSteps; ++st) {
                const uint32_t rec = st * kRecords + record;
                const uint32_t i = __shfl(index[a], static_cast<int>(rec & 63u));
                w[a][st] = 0u;
                if (record < kRecords && rec < 64 && t0 + a * 64 + rec < total && i < rows) {
                    w[a][st] = column[static_cast<size_t>(i) * units];
                }
            }
        }
#pragma unroll
        for (int a = 0; a < kSortAhead; ++a) {
#pragma unroll
            for (int st = 0; st < kSteps; ++st) {
                const uint32_t rec = st * kRecords + record;
                const uint32_t to = __shfl(at[a], static_cast<int>(rec & 63u));
                if (record < kRecords && rec < 64 && t0 + a * 64 + rec < total) {
                    sort.rows[static_cast<size_t>(to) * WORDS + word] = w[a][st];
                }
            }
        }
    }
}

// Pass 3: a chunk's rows to its queries.
constexpr int kDealThreads = 1024;

__global__ __launch_bounds__(kDealThreads) void deal_rows_kernel(RowTables tabs, RowSort sort, int miss_row) {
    extern __shared__ __align__(16) uint32_t s_rows[];   // kSortChunk * words, and the places
    uint16_t* s_place = reinterpret_cast<uint16_t*>(s_rows + kSortChunk * sort.words);
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kSortChunk;
    const uint32_t queries = sort.n - base < kSortChunk ? static_cast<uint32_t>(sort.n - base) : kSortChunk;
    const uint16_t* bounds = sort.bounds + static_cast<int64_t>(blockIdx.x) * kSortBounds;
    if (bounds[kSortParts + 1] == kBoundsServed) return;
    const uint32_t found = bounds[kSortParts], total = found * sort.words;
    const uint32_t* rows = sort.rows + static_cast<size_t>(base) * sort.words;
    // (whole pieces: a chunk's region is kSortChunk rows long.  Read once, and marked so:
    // 100 -> 96 us for 16 M rows of 16 bytes.  Pass 2's indices marked like this cost it
    // 274 -> 296, its rows 315: what it reads and writes a line of, others touch as well)
    typedef uint32_t v4u __attribute__((ext_vector_type(4)));
    for (uint32_t t = threadIdx.x; t < (total + 3) / 4; t += kDealThreads) {
        reinterpret_cast<v4u*>(s_rows)[t] = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(rows) + t);
    }
    for (uint32_t t = threadIdx.x; t < queries; t += kDealThreads) s_place[t] = sort.place[base + t];
    __syncthreads();
    if (bounds[kSortParts + 1] == kBoundsLong) {
        // rows that pass 2 has left: queries that crowd in few parts, and so in the caches
        for (uint32_t t = threadIdx.x; t < found; t += kDealThreads) {
            const int32_t kept = sort.index[base + t];
            if (kept >= 0) continue;
            const uint32_t index = static_cast<uint32_t>(~kept);
            uint32_t* row = s_rows + t * sort.words;
            for (int v = 0; v < tabs.n; ++v) {
                const uint32_t units = tabs.units[v];
                const uint32_t* src = static_cast<const uint32_t*>(tabs.src[v]) + static_cast<size_t>(index) * units;
                for (uint32_t u = 0; u < units; ++u) row[u] = index < tabs.src_rows[v] ? src[u] : 0u;
                row += units;
            }
        }
        __syncthreads();
    }
    uint32_t column = 0;
    for (int v = 0; v < tabs.n; ++v) {
        const uint32_t units = tabs.units[v], magic = tabs.magic[v];
        uint32_t* out = static_cast<uint32_t*>(tabs.dst[v]) + static_cast<size_t>(base) * units;
        const bool miss_reads = miss_row >= 0 && static_cast<uint32_t>(miss_row) < tabs.src_rows[v];
        for (uint32_t t = threadIdx.x; t < queries * units; t += kDealThreads) {
            const uint32_t q = units == 1 ? t : __umulhi(t, magic);
            const uint32_t word = t - q * units;
            const uint32_t place = s_place[q];
            uint32_t w = 0u;
            if (place != kNoPlace) {
                w = s_rows[place * sort.words + column + word];
            } else if (miss_reads) {
                w = static_cast<const uint32_t*>(tabs.src[v])[static_cast<size_t>(miss_row) * units + word];
            }
            __builtin_nontemporal_store(w, out + t);
        }
        column += units;
    }
}

// 16 bytes per thread, the words of a shorter tail one by one.
__global__ __launch_bounds__(kBlock) void clear_rows_kernel(uint32_t* __restrict__ p, int64_t words) {
    const int64_t t = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) * 4;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock * 4;
    for (int64_t at = t; at < words; at += stride) {
        if (at + 4 <= words) {
            *reinterpret_cast<uint4*>(p + at) = make_uint4(0u, 0u, 0u, 0u);
        } else {
            for (int64_t w = at; w < words; ++w) p[w] = 0u;
        }
    }
}

// out[indices[i]] += rows[i] where masks[i]: the transpose of the look-up.  One
// element per thread, so that the elements of a row leave in one atomic request
// per 64-byte line whatever the row's width; the device executes such requests
// at 15-20 G/s, which is what bounds this kernel (200 003 rows of 16 floats:
// 13 us, where sorting the indices and adding the rows up in order took 8.8 ms).
template <typename T>
__global__ __launch_bounds__(kBlock) void add_rows_kernel(
        const T* __restrict__ rows, const int64_t* __restrict__ indices,
        const uint8_t* __restrict__ masks, int64_t n, int64_t width, T* __restrict__ out,
        int64_t out_rows) {
    const int64_t total = n * width;
    const bool narrow = total <= 0xFFFFFFFFll;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock;
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; t < total; t += stride) {
        const int64_t row = narrow ? static_cast<int64_t>(static_cast<uint32_t>(t) /
                                                          static_cast<uint32_t>(width))
                                   : t / width;
        const int64_t to = indices[row];
        if (masks[row] == 0 || to < 0 || to >= out_rows) continue;
        unsafeAtomicAdd(out + to * width + (t - row * width), rows[t]);
    }
}

// The rows whose flag an activation has set, in ascending order, with their
// block coordinates; the flags are cleared on the way and the count goes to
// the table's counters, where the read-back that follows an activation finds
// it (and where ash_grid_integrate_depth_touched reads it on the device).
//
// Up to kCollectGroups workgroups, each with a chunk of the flags: a workgroup
// holds its own chunk in registers (one run of `words` 4-flag words per thread,
// so that thread order is flag order), counts the flags of all chunks before
// its own (they sit in L2: every workgroup reads them) and so knows where its
// rows go without waiting for anybody.  Nobody may clear flags while others
// still count them: each workgroup draws a ticket when it has read all it
// needs, and the one that draws the last ticket clears the whole array and
// puts the ticket counter back to zero.
constexpr int kCollectThreads = 1024;
constexpr int kCollectGroups = 128;
constexpr int kCollectMaxWords = 2;    // per thread: 2^20 flags / 128 groups / 1024 threads / 4
constexpr int64_t kCollectMaxBlocks = int64_t{1} << 20;   // ASH_COLLECT_MAX_BLOCKS of the header
constexpr int64_t kCountFlags = int64_t{1} << 18;   // per workgroup of count_flags_kernel: 16 loads a thread

__device__ __forceinline__ int flags_in(uint32_t w) {
    return (w & 0xFFu ? 1 : 0) + (w & 0xFF00u ? 1 : 0) + (w & 0xFF0000u ? 1 : 0) +
           (w & 0xFF000000u ? 1 : 0);
}

// word `i` of the flags, bytes beyond `capacity` read as zero
__device__ __forceinline__ uint32_t flag_word(const uint8_t* touched, int64_t i, int64_t capacity) {
    const int64_t at = i * 4;
    if (at + 4 <= capacity) return *reinterpret_cast<const uint32_t*>(touched + at);
    uint32_t w = 0;
    for (int b = 0; at + b < capacity; ++b) w |= static_cast<uint32_t>(touched[at + b]) << (8 * b);
    return w;
}

// Sum of `v` over the workgroup; `mine` = sum over the threads before this one.
__device__ __forceinline__ int block_sums(int v, int* s_wave, int& mine) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    int incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int up = __shfl_up(incl, d);
        if (lane >= d) incl += up;
    }
    __syncthreads();   // s_wave free again
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    mine = incl - v;
    int total = 0;
    for (int q = 0; q < kCollectThreads / 64; ++q) {
        if (q < wave) mine += s_wave[q];
        total += s_wave[q];
    }
    return total;
}

// The counters for the host, `total` blocks touched among them (one workgroup).
__device__ __forceinline__ void leave_touched(int32_t* ctr, int total, uint64_t* landing,
                                              int32_t stamp) {
    if (threadIdx.x < kHostCounters) {
        const int32_t v = threadIdx.x == kCtrTouched ? total : ctr[threadIdx.x];
        if (threadIdx.x == kCtrTouched) ctr[kCtrTouched] = total;
        leave_word(landing + threadIdx.x, v, stamp);
    }
}

// How many of the first `rows` rows are flagged, while the flags stand: `counts[w]`
// of workgroup w's share, and where one workgroup looks at all of them the counters
// go to the host at once.  The flags are read 16 at a time, eight loads of a thread
// on their way together (80 000 flags are five loads each: one wait for memory).
__global__ __launch_bounds__(kCollectThreads) void count_flags_kernel(
        const uint8_t* __restrict__ touched, int64_t rows, int32_t* __restrict__ counts,
        int32_t* __restrict__ ctr, uint64_t* landing, int32_t stamp) {
    __shared__ int s_wave[kCollectThreads / 64];
    const int64_t at = static_cast<int64_t>(blockIdx.x) * kCollectThreads + threadIdx.x;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kCollectThreads;
    // what lies before the first whole 16 bytes and behind the last is counted byte by byte
    int64_t head = (16 - static_cast<int64_t>(reinterpret_cast<uintptr_t>(touched) % 16)) % 16;
    if (head > rows) head = rows;
    const int64_t whole = (rows - head) / 16;
    const uint4* quads = reinterpret_cast<const uint4*>(touched + head);
    int sum = 0;
#pragma unroll 8
    for (int64_t i = at; i < whole; i += stride) {
        const uint4 v = quads[i];
        sum += flags_in(v.x) + flags_in(v.y) + flags_in(v.z) + flags_in(v.w);
    }
    if (at < head) sum += touched[at] != 0;
    const int64_t rest = head + whole * 16 + at;
    if (rest < rows) sum += touched[rest] != 0;
    int unused;
    const int total = block_sums(sum, s_wave, unused);
    if (gridDim.x > 1) {
        if (threadIdx.x == 0) counts[blockIdx.x] = total;
        return;
    }
    leave_touched(ctr, total, landing, stamp);
}

// The same for several workgroups: their counts added up (one workgroup).
__global__ __launch_bounds__(kCollectThreads) void publish_touched_kernel(
        int32_t* __restrict__ ctr, const int32_t* __restrict__ counts, int n, uint64_t* landing,
        int32_t stamp) {
    __shared__ int s_wave[kCollectThreads / 64];
    int sum = 0;
    for (int i = threadIdx.x; i < n; i += kCollectThreads) sum += counts[i];
    int unused;
    const int total = block_sums(sum, s_wave, unused);
    leave_touched(ctr, total, landing, stamp);
}

__global__ __launch_bounds__(kCollectThreads) void collect_touched_kernel(
        uint8_t* __restrict__ touched, const int32_t* __restrict__ block_coords,
        int64_t capacity, int words, int64_t* __restrict__ out_idx,
        int32_t* __restrict__ out_coords, int32_t* __restrict__ ctr) {
    __shared__ int s_wave[kCollectThreads / 64];
    __shared__ int s_last;
    const int64_t chunk_words = static_cast<int64_t>(words) * kCollectThreads;
    const int64_t first_word = blockIdx.x * chunk_words + static_cast<int64_t>(threadIdx.x) * words;
    uint32_t w[kCollectMaxWords];
    int own = 0;
#pragma unroll
    for (int i = 0; i < kCollectMaxWords; ++i) {
        w[i] = i < words ? flag_word(touched, first_word + i, capacity) : 0u;
        own += flags_in(w[i]);
    }
    int before = 0;
    const int64_t words_before = blockIdx.x * chunk_words;   // whole words, inside the array
    if (reinterpret_cast<uintptr_t>(touched) % 16 == 0) {
        const uint4* quads = reinterpret_cast<const uint4*>(touched);
#pragma unroll 8
        for (int64_t i = threadIdx.x; i < words_before / 4; i += kCollectThreads) {
            const uint4 v = quads[i];
            before += flags_in(v.x) + flags_in(v.y) + flags_in(v.z) + flags_in(v.w);
        }
    } else {
#pragma unroll 8
        for (int64_t i = threadIdx.x; i < words_before; i += kCollectThreads) {
            before += flags_in(reinterpret_cast<const uint32_t*>(touched)[i]);
        }
    }
    int unused;
    const int base = block_sums(before, s_wave, unused);
    int pos;
    const int total = block_sums(own, s_wave, pos);
    pos += base;
    if (threadIdx.x == 0) {
        if (blockIdx.x == gridDim.x - 1) ctr[kCtrTouched] = base + total;
        __threadfence();
        s_last = atomicAdd(ctr + kCtrTicket, 1) == static_cast<int>(gridDim.x) - 1;
    }
#pragma unroll
    for (int i = 0; i < kCollectMaxWords; ++i) {
        if (w[i] == 0u) continue;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            if ((w[i] >> (8 * b)) & 0xFFu) {
                const int64_t at = (first_word + i) * 4 + b;
                out_idx[pos] = at;
                out_coords[pos * 3 + 0] = block_coords[at * 3 + 0];
                out_coords[pos * 3 + 1] = block_coords[at * 3 + 1];
                out_coords[pos * 3 + 2] = block_coords[at * 3 + 2];
                ++pos;
            }
        }
    }
    __syncthreads();
    if (!s_last) return;
    // every workgroup has read what it needs
    const int64_t whole = capacity / 4;
    for (int64_t i = threadIdx.x; i < whole; i += kCollectThreads) {
        reinterpret_cast<uint32_t*>(touched)[i] = 0u;
    }
    if (threadIdx.x < capacity - whole * 4) touched[whole * 4 + threadIdx.x] = 0;
    if (threadIdx.x == 0) ctr[kCtrTicket] = 0;
}

// Puts the entries of the packed region back into an emptied bucket array:
// entry i of the key log is the code stored under index i.  `identity`: only
// the entries below the size are in use (see items_kernel).
__global__ __launch_bounds__(kHeapBlock) void replace_from_log_kernel(MapDev m, int identity) {
    const int64_t limit = identity ? static_cast<int64_t>(m.ctr[kCtrSize])
                                   : static_cast<int64_t>(m.capacity);
    const ValueArgs none = {};
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kHeapBlock;
    for (int64_t first = static_cast<int64_t>(blockIdx.x) * kHeapBlock; first < limit;
         first += stride) {
        const int64_t i = first + threadIdx.x;
        const uint64_t code = i < limit ? m.klog[i] : kEmpty;
        const int32_t k[1] = {0};
        insert_key<1, kInsertLoad, false>(m, k, code, true, i, code < kTomb, none, nullptr, nullptr);
    }
}

// Entries of a heap that address no row, counted with the pairs a load refuses.
// Inserts write to the rows and log entries that they draw from the heap; from one
// with such entries nothing is drawn: it counts as exhausted until a clear or a load.
__global__ __launch_bounds__(kBlock) void check_heap_kernel(const int32_t* __restrict__ heap,
                                                           int64_t capacity,
                                                           int32_t* __restrict__ ctr) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock;
    int bad = 0;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < capacity;
         i += stride) {
        bad += static_cast<uint32_t>(heap[i]) >= static_cast<uint32_t>(capacity) ? 1 : 0;
    }
    if (bad) {
        atomicAdd(ctr + kCtrLoadDup, bad);
        atomicMax(ctr + kCtrSize, static_cast<int32_t>(capacity));
    }
}

// ---------------------------------------------------------------- host
inline unsigned grid_for(int64_t n, int per_block = kBlock) {
    return static_cast<unsigned>((n + per_block - 1) / per_block);
}

// One unit per thread as far as a launch goes (the kernels loop beyond that):
// workgroups that are handed out one after the other walk through memory in
// order, which the memory side rewards (a 1.6 GB fill: 6.8 TB/s, against 5.7
// with 16 384 workgroups that stride through it and 4.5 with 4096).
inline unsigned capped_grid(int64_t n) {
    int64_t g = (n + kBlock - 1) / kBlock;
    const int64_t cap = 0x7FFFFFFF;
    if (g > cap) g = cap;
    if (g < 1) g = 1;
    return static_cast<unsigned>(g);
}

// For the kernels that move rows by index (random on one side): 8192
// workgroups that loop (one unit per thread: 0.23 against 0.185 ms for the 16 M
// rows of two value tensors).
inline unsigned looping_grid(int64_t n) {
    int64_t g = (n + kBlock - 1) / kBlock;
    const int64_t cap = 256 * 32;
    if (g > cap) g = cap;
    if (g < 1) g = 1;
    return static_cast<unsigned>(g);
}

int check_map(const ash_map* map) {
    if (map == nullptr) ASH_FAIL("null map handle");
    return 0;
}

// Whether no entry lives in the second region: there is none, or the counters as
// the host knows them say that it is empty.
bool none_in_general(ash_map* map) {
    if (!map->general_attached) return true;
    std::lock_guard<std::mutex> lock(map->counter_lock);
    return map->counters_known && map->counters.general_live == 0;
}

// Whether a listing has entry i under index i: nothing has written to the heap
// since it was last 0, 1, 2, ... (no erase, no load) and no entry lives in the
// second region.
bool lists_in_index_order(ash_map* map) { return heap_in_order(map) && none_in_general(map); }

int fill_buckets(ash_map* map, hipStream_t s) {
    const int64_t n16 = static_cast<int64_t>(map->d.nb) * kGroup;
    fill16_kernel<<<capped_grid(n16), kBlock, 0, s>>>(
            reinterpret_cast<uint4*>(map->d.buckets), n16, 0xFFFFFFFFu);
    ASH_LAUNCH_CHECK();
    map->table_stale = map->table_filled = false;
    return 0;
}

// Empties the table and sets the size to `size`.
int clear_table(ash_map* map, hipStream_t s, bool write_heap, int32_t size) {
    if (fill_buckets(map, s)) return 1;
    if (map->general_attached) {
        const int64_t g16 = static_cast<int64_t>(map->d.gslots) / 4;
        fill16_kernel<<<capped_grid(g16), kBlock, 0, s>>>(
                reinterpret_cast<uint4*>(map->d.gstate), g16, 0xFFFFFFFFu);
        ASH_LAUNCH_CHECK();
    }
    // The key log: every index is free again.  While nothing has written to the
    // heap since its last reset the indices in use are 0 .. size-1 and nothing
    // reads the log beyond the size: that part of the log (read on the device,
    // before the counters are reset below) is emptied, or all of it once the heap
    // has been written to.
    const int64_t n16 = (map->capacity + 1) / 2;
    // (a prefix of unknown length: few workgroups that loop, not one per
    // 4 KB of the capacity, most of which would start only to leave)
    empty_log_kernel<<<map->heap_dirty ? capped_grid(n16) : looping_grid(n16), kBlock, 0, s>>>(
            reinterpret_cast<uint4*>(map->d.klog), map->capacity, map->d.ctr,
            map->heap_dirty ? 0 : 1);
    ASH_LAUNCH_CHECK();
    map->log_stale = false;
    // Inserts only read the heap; while nothing has written to it since the
    // last reset it still is 0, 1, 2, ... and only the counters are reset.
    const bool rewrite = write_heap && map->heap_dirty;
    int64_t span = rewrite && map->capacity > kNumCounters ? map->capacity : kNumCounters;
    reset_heap_kernel<<<grid_for(span), kBlock, 0, s>>>(
            map->d.heap, map->capacity, map->d.ctr, size, rewrite);
    ASH_LAUNCH_CHECK();
    if (rewrite) map->heap_dirty = false;
    return 0;
}

// Value rows that a clear zeroes along with the table (16-byte aligned).
struct ClearRows {
    int n;
    void* const* rows;
    const int64_t* bytes;
};

class ClearList {
  public:
    void add(void* p, int64_t bytes, uint32_t word, bool count = false) {
        if (bytes <= 0) return;
        const int64_t pieces = bytes / 16;
        args_.span[args_.n++] = {static_cast<uint4*>(p), pieces, word, static_cast<uint8_t>(bytes % 16),
                                 count, static_cast<uint32_t>(groups_)};
        groups_ += (pieces + (bytes % 16 != 0 ? 1 : 0) + kBlock - 1) / kBlock;
    }
    void add(const ClearRows& rows) {
        for (int v = 0; v < rows.n; ++v) add(rows.rows[v], rows.bytes[v], 0u);
    }
    int launch(const ash_map* map, int counters, bool keep_log, hipStream_t s) const {
        if (groups_ > 0x7FFFFFFF) ASH_FAIL("too many bytes to clear in one call");
        if (groups_ == 0 && counters == kCountersAsTheyAre) return 0;
        clear_kernel<<<static_cast<unsigned>(groups_ > 0 ? groups_ : 1), kBlock, 0, s>>>(
                args_, map->d.ctr, counters, keep_log);
        ASH_LAUNCH_CHECK();
        return 0;
    }

  private:
    ClearArgs args_ = {};
    int64_t groups_ = 0;
};

// What a clear does of a map whose state the host knows, and what makes a new one
// (`fresh`): counters, heap and second region are reset at once.  The bucket array is
// left to the next call that needs it (settle_table) -- a streaming insert writes
// every bucket itself -- unless the table is so small that it is filled here, without
// a launch of its own (kFillAtOnce).  The key log is left
// alone while the heap is in its initial order (no listing reads an entry beyond the
// size then), or emptied with the heap's order.
int clear_lazily(ash_map* map, hipStream_t s, bool fresh, const ClearRows& rows) {
    ClearList list;
    list.add(rows);
    const bool small = static_cast<int64_t>(map->d.nb) <= kFillAtOnce;
    if (small) list.add(map->d.buckets, static_cast<int64_t>(map->d.nb) * kGroup * 16, ~0u);
    if (map->general_attached) list.add(map->d.gstate, static_cast<int64_t>(map->d.gslots) * 4, ~0u);
    const bool keep_log = !map->heap_dirty;
    const bool wide = reinterpret_cast<uintptr_t>(map->d.heap) % 16 == 0;   // (the caller's own buffer)
    if (!keep_log) {
        list.add(map->d.klog, (map->capacity + 1) / 2 * 16, ~0u);
        if (wide) list.add(map->d.heap, map->capacity * 4, 0u, true);
    }
    if (list.launch(map, fresh ? kCountersFresh : kCountersReset, keep_log, s)) return 1;
    if (!keep_log && !wide) {
        reset_heap_kernel<<<grid_for(std::max<int64_t>(map->capacity, kNumCounters)), kBlock, 0, s>>>(
                map->d.heap, map->capacity, map->d.ctr, 0, true);
        ASH_LAUNCH_CHECK();
    }
    map->table_stale = true;
    map->table_filled = small;
    map->log_stale = keep_log;
    map->heap_dirty = false;
    return 0;
}

}  // namespace

// ------------------------------------------- words that the device leaves here
// What the host wants to know of a running call (the counters, how many keys the
// first pass of a streaming insert could not place) is written by kernels into
// page-locked host memory, stamped with a number of the call's own, and the host
// polls the stamp: no copy on the stream, no event, and the answer is seen about
// a microsecond after it was written, where a copy and a stream synchronisation
// took 12-15 us of an idle device's time.
//
// A call that waits takes a line of kLineWords for itself and returns it (two
// threads that read one map's counters have one each), and a map keeps one from
// its first streaming insert or counted frame until it is destroyed.  The pool
// serves the process: as many lines as were ever in use at the same time.
namespace {

constexpr int kLinesPerSlab = 64;

std::mutex g_lines_mutex;
std::vector<uint64_t*>& free_lines() {
    static auto* lines = new std::vector<uint64_t*>;   // (outlives maps destroyed at exit)
    return *lines;
}

int take_free_line(uint64_t** line) {
    std::lock_guard<std::mutex> lock(g_lines_mutex);
    std::vector<uint64_t*>& lines = free_lines();
    if (lines.empty()) {
        void* slab = nullptr;
        ASH_HIP(hipHostMalloc(&slab, kLinesPerSlab * kLineWords * sizeof(uint64_t),
                              hipHostMallocPortable | hipHostMallocCoherent));
        memset(slab, 0, kLinesPerSlab * kLineWords * sizeof(uint64_t));
        for (int i = 0; i < kLinesPerSlab; ++i) {
            lines.push_back(static_cast<uint64_t*>(slab) + i * kLineWords);
        }
    }
    *line = lines.back();
    lines.pop_back();
    return 0;
}

// (no launch may still owe words there)
void give_back_line(uint64_t* line) {
    if (line == nullptr) return;
    std::lock_guard<std::mutex> lock(g_lines_mutex);
    free_lines().push_back(line);
}

int32_t next_stamp(int32_t stamp) {   // (2^31 - 1 goes on at -2^31)
    return static_cast<int32_t>(static_cast<uint32_t>(stamp) + 1u);
}

// The stamp at which the owners of a line so far have stopped: the latest has left
// it in a place's first word.
int32_t stamp_of_line(const uint64_t* line) {
    return std::max(stamp_of(line[kLineLate]), stamp_of(line[kLineEarly]));
}

bool all_come(const uint64_t* words, int count, int32_t stamp) {
    for (int w = 0; w < count; ++w) {
        if (stamp_of(__atomic_load_n(words + w, __ATOMIC_ACQUIRE)) != stamp) return false;
    }
    return true;
}

// Looks for `count` words under `stamp` `looks` times, 20 - 50 ns apart; true: they
// have come.
bool has_come(const uint64_t* words, int count, int32_t stamp, int looks) {
    for (int look = 0; look < looks; ++look) {
        if (all_come(words, count, stamp)) return true;
        __builtin_ia32_pause();
    }
    return all_come(words, count, stamp);
}

}  // namespace

int Answer::take() {
    if (take_free_line(&words)) return 1;
    stamp = next_stamp(stamp_of_line(words));
    return 0;
}

// Looks for the words for some ten milliseconds.  Where work that takes longer is
// queued ahead the stream, of which the launch that leaves them is the last, is
// waited for (which keeps a core just as busy and comes back 5 us later); errors
// show there, and the words have to be there afterwards.
int Answer::wait(hipStream_t s, int count) {
    lost_ = true;
    if (!has_come(words, count, stamp, 400'000)) {
        ASH_HIP(hipStreamSynchronize(s));
        if (!has_come(words, count, stamp, 1)) ASH_FAIL("internal error: the device has not left its answer");
    }
    lost_ = false;
    return 0;
}

Answer::~Answer() {
    if (!lost_) give_back_line(words);
}

int take_line(ash_map* map) {
    std::lock_guard<std::mutex> lock(map->counter_lock);
    if (map->line != nullptr) return 0;
    if (take_free_line(&map->line)) return 1;
    map->stamp = stamp_of_line(map->line);
    return 0;
}

// Waits until the device has left `count` words under `stamp` with more work queued
// behind the launch that does: an event there would cost 3 of the 75 us of a set of
// 1 M keys, the stream's end comes too late for what is to be queued next, and the
// stream may be gone.  Where more than a short call is queued ahead, the words are
// looked for every tenth of a millisecond (no core is kept busy and no other stream
// waited for); only when a minute has passed the device is synchronised, where
// an error would show.
int wait_for_words(const uint64_t* words, int count, int32_t stamp) {
    bool come = has_come(words, count, stamp, 20'000);
    for (int look = 0; !come && look < 600'000; ++look) {
        std::this_thread::sleep_for(std::chrono::microseconds(100));
        come = all_come(words, count, stamp);
    }
    if (come) return 0;
    ASH_HIP(hipDeviceSynchronize());
    if (!has_come(words, count, stamp, 1)) ASH_FAIL("internal error: the device has not left its counters");
    return 0;
}

namespace {

// A read-back queued behind an insert that may still be under way has to arrive
// before its words are read or written again.  The caller holds the map's
// counter_lock.
int settle_late_words(ash_map* map) {
    if (map->late_in_flight) {
        if (wait_for_words(map->line + kLineLate, kHostCounters, map->late_stamp)) return 1;
        map->late_in_flight = false;
    }
    return 0;
}

void decode_counters(const uint64_t* words, ash_counters& c) {
    int32_t host[kHostCounters];
    for (int w = 0; w < kHostCounters; ++w) host[w] = value_of(words[w]);
    c.size = host[kCtrSize];
    c.dropped = host[kCtrDropped];
    c.tombstones = host[kCtrTombs];
    c.exotic_pending = host[kCtrExotic];
    c.load_refused = host[kCtrLoadDup];
    c.touched = host[kCtrTouched];
    c.general_live = host[kCtrGenLive];
    c.general_tombstones = host[kCtrGenTombs];
}

// map->counters are those of the device.  The caller holds the map's counter_lock.
void counters_taken(ash_map* map) {
    map->counters_known = true;
    map->unread_inserts = 0;
    if (map->counters.dropped > 0 || map->counters.tombstones > 0) map->maybe_tombstones = true;
}

// The words that a call has queued, if they are the latest state, waited for and
// taken.  The caller holds the map's counter_lock.
int take_late_words(ash_map* map) {
    if (!map->late_pending) return 0;
    if (settle_late_words(map)) return 1;
    map->late_pending = false;
    decode_counters(map->line + kLineLate, map->counters);
    counters_taken(map);
    return 0;
}

// The map's own words, for the call that changes the map (there is one at a time): what
// earlier calls owe there has come when they are taken.  A call that ends between its
// launches and `queued` or `unused` may owe words itself: the line is given up then
// (128 bytes), and the next call takes another.
class LatePlace {
  public:
    explicit LatePlace(ash_map* map) : map_(map) {}
    LatePlace(const LatePlace&) = delete;
    LatePlace& operator=(const LatePlace&) = delete;
    ~LatePlace() {
        if (!taken_) return;
        std::lock_guard<std::mutex> lock(map_->counter_lock);
        map_->line = nullptr;
        map_->late_in_flight = map_->late_pending = false;
    }
    // `settle`: words that are owed are waited for; else the place may not be had.
    int take(bool settle) {
        if (take_line(map_)) return 1;
        std::lock_guard<std::mutex> lock(map_->counter_lock);
        if (!settle && map_->late_in_flight &&
            !all_come(map_->line + kLineLate, kHostCounters, map_->late_stamp)) {
            return 0;
        }
        if (take_late_words(map_) || settle_late_words(map_)) return 1;
        stamp = map_->stamp = next_stamp(map_->stamp);
        taken_ = true;
        return 0;
    }
    bool taken() const { return taken_; }
    uint64_t* late() const { return map_->line + kLineLate; }
    uint64_t* early() const { return map_->line + kLineEarly; }
    // The launch that leaves the counters at `late` under `stamp` is queued, the last
    // of its Change: they are the latest state.
    void queued(bool of_erase = false) {
        std::lock_guard<std::mutex> lock(map_->counter_lock);
        taken_ = false;
        map_->late_stamp = stamp;
        map_->late_in_flight = map_->late_pending = true;
        map_->late_of_erase = of_erase;
        map_->counters_known = false;   // (a reader may have asked the device since)
        if (!of_erase) map_->unread_inserts = 0;
    }
    // No launch leaves words any more.
    void unused() { taken_ = false; }
    int32_t stamp = 0;

  private:
    ash_map* map_;
    bool taken_ = false;
};

}  // namespace

namespace {

int32_t* next_ticket(ash_map* map) { return map->d.ctr + kCtrTickets + next_slot(map); }

// Keys up to which a launch leaves the counters itself (leave_with_last), instead
// of one of its own behind it.  Its tickets queue on the line of the counters.  A call
// and the size after it, own launch -> left (us): insert of 200 keys 18.4 -> 18.0,
// 65 000 23.8 -> 22.6, 131 000 30.0 -> 30.3, 262 000 48 -> 50, 1 M 98 -> 108; erase
// 13.4 -> 12.9, 16.9 -> 16.3, 20.0 -> 19.1, 32 -> 30, 64.7 -> 66.5.  With work queued
// in between a launch less counts 4 us.
constexpr int64_t kLeaveKeys = int64_t{1} << 17;

}  // namespace

int give_up_heap_order(ash_map* map, hipStream_t s) {
    if (map->heap_dirty) return 0;
    map->heap_dirty = true;
    if (!map->log_stale) return 0;
    empty_log_tail_kernel<<<looping_grid(map->capacity), kBlock, 0, s>>>(
            map->d.klog, map->capacity, map->d.ctr);
    ASH_LAUNCH_CHECK();
    map->log_stale = false;
    return 0;
}

namespace {

template <int MODE, bool TOMBS, int BLOCK, bool ALONE>
int launch_insert_by(ash_map* map, const int32_t* keys, int64_t n,
                     const ValueArgs& va, int32_t* assigned, const int64_t* given,
                     hipStream_t s, const Publish& publish = {}, const KeyCheck& check = {}) {
    const unsigned g = grid_for(n, BLOCK) + check.groups;
    auto kernel = map->key_dim == 1   ? insert_kernel<1, MODE, TOMBS, BLOCK, ALONE>
                  : map->key_dim == 2 ? insert_kernel<2, MODE, TOMBS, BLOCK, ALONE>
                  : map->key_dim == 3 ? insert_kernel<3, MODE, TOMBS, BLOCK, ALONE>
                                      : insert_kernel<4, MODE, TOMBS, BLOCK, ALONE>;
    kernel<<<g, BLOCK, 0, s>>>(map->d, keys, n, va, assigned, given, publish, check);
    ASH_LAUNCH_CHECK();
    return 0;
}

// Larger workgroups update the heap counter (and, of tombstones, theirs) less often, but
// each of their wavefronts waits for the slowest probe of all.  A batch that comes, is read
// and goes, of 256 -> 512 threads (us): 140 000 keys beside 20 000 111 -> 115, beside a
// million 116 -> 114; 200 000 beside a million 135 -> 128, beside four 225 -> 217; 400 000
// beside 300 000 188 -> 162; a million beside four 424 -> 397 (1024 threads: 402).
//
// Every lane looks at its buckets by itself, which takes half of the
// vector instructions and registers (the kernel with rows of 16 bytes, cooperative ->
// alone, beside a million keys: 8000 12.5 -> 11.3 us, 65 537 20.8 -> 19.3, 131 000 29.5 ->
// 27.0, 300 000 39 -> 34; beside 100 000 131 000 36.8 -> 31.7, 196 000 48.6 -> 39; keys
// alone into an emptied table 16 000 13.1 -> 11.7, 98 000 21.8 -> 20.3).  Keys that are
// stored already gain as well, beyond where look-ups (kAloneKeys) do not: beside 100 000 | four million | sixteen, a million 19.6 -> 17.4 | 25.0 -> 23.5 | 27.4 -> 24.3, 3.1
// million 52.5 -> 45.9 | 64.0 -> 62.7 | 70 -> 63; of new keys, each sixteen times, a million
// 36 -> 33 | 37 -> 35 | 42 -> 37, 3.1 million 82 -> 77 | 90 -> 80 | 95 -> 80; half stored, half
// new 50 -> 45 | 52 -> 50 | 56 -> 52, 129 -> 126 | 180 -> 169 | 188 -> 165. Larger
// batches, 256 cooperative -> 512 alone, of new keys: with rows of 4 bytes four million beside
// four 285 -> 254, eight beside eight 532 -> 492, five beside sixteen 337 -> 297, of 16 bytes
// sixteen beside sixteen 573 -> 556; keys alone 3.5 million beside four 242 -> 208, each
// sixteen times 114 -> 83; stored ones 127 -> 131, eight million 253 -> 253.  (While all keys
// of a bucket went for its first free slot, see first_slot, four million were slower alone.)
// Loads, 256 threads: 3000 keys 8.2 -> 6.9, 30 000 12.1 -> 10.8, 300 000 33.7 -> 25.9, a
// million 80 -> 58, two 130 -> 122, three 225 -> 233, four 306 -> 312, sixteen 931 -> 1042.
constexpr int64_t kWideInsert = int64_t{3} << 16, kAloneLoad = int64_t{1} << 21;
constexpr int kWideBlock = 512;

template <int MODE, bool TOMBS>
int launch_insert_to(ash_map* map, const int32_t* keys, int64_t n,
                     const ValueArgs& va, int32_t* assigned, const int64_t* given,
                     hipStream_t s, const Publish& publish = {}, const KeyCheck& check = {}) {
    if constexpr (MODE == kInsertKeys || MODE == kInsertFused) {
        return n > kWideInsert
                       ? launch_insert_by<MODE, TOMBS, kWideBlock, true>(map, keys, n, va, assigned, given, s, publish, check)
                       : launch_insert_by<MODE, TOMBS, kHeapBlock, true>(map, keys, n, va, assigned, given, s, publish, check);
    } else {
        if constexpr (MODE == kInsertLoad) {
            if (n <= kAloneLoad) {
                return launch_insert_by<MODE, TOMBS, kHeapBlock, true>(map, keys, n, va, assigned, given, s, publish, check);
            }
        }
        return launch_insert_by<MODE, TOMBS, kHeapBlock, false>(map, keys, n, va, assigned, given, s, publish, check);
    }
}

template <int MODE>
int launch_insert(ash_map* map, const int32_t* keys, int64_t n,
                  const ValueArgs& va, int32_t* assigned, const int64_t* given,
                  hipStream_t s, const Publish& publish, const KeyCheck& check) {
    return tombs_in(map)
                   ? launch_insert_to<MODE, true>(map, keys, n, va, assigned, given, s, publish, check)
                   : launch_insert_to<MODE, false>(map, keys, n, va, assigned, given, s, publish, check);
}

template <int MODE, bool TOMBS>
int launch_selected_to(ash_map* map, bool codes, const int32_t* keys,
                       const int32_t* sel, const int32_t* nsel,
                       const ValueArgs& va, hipStream_t s, const Publish& publish) {
    // the selection is empty or short as a rule: a grid that costs little to
    // launch, whose workgroups stride over a long one
    constexpr unsigned g = 128;
    auto kernel = codes               ? insert_selected_kernel<1, MODE, TOMBS, true>
                  : map->key_dim == 1 ? insert_selected_kernel<1, MODE, TOMBS, false>
                  : map->key_dim == 2 ? insert_selected_kernel<2, MODE, TOMBS, false>
                  : map->key_dim == 3 ? insert_selected_kernel<3, MODE, TOMBS, false>
                                      : insert_selected_kernel<4, MODE, TOMBS, false>;
    kernel<<<g, kHeapBlock, 0, s>>>(map->d, keys, sel, nsel, va, publish);
    ASH_LAUNCH_CHECK();
    return 0;
}

template <int MODE>
int launch_selected(ash_map* map, bool codes, const int32_t* keys,
                    const int32_t* sel, const int32_t* nsel,
                    const ValueArgs& va, hipStream_t s, const Publish& publish) {
    return tombs_in(map) ? launch_selected_to<MODE, true>(map, codes, keys, sel, nsel, va, s, publish)
                         : launch_selected_to<MODE, false>(map, codes, keys, sel, nsel, va, s, publish);
}

}  // namespace

namespace {

// The tables of a gather, checked, and the words of the one with most of them for
// n rows.
int gather_args(int n_values, const void* const* src, void* const* dst, const int64_t* row_bytes,
                const int64_t* src_rows, int64_t n, GatherArgs& a, int64_t& most) {
    if (src == nullptr || dst == nullptr || row_bytes == nullptr || src_rows == nullptr) {
        ASH_FAIL("null value tables");
    }
    a = {};
    a.n = n_values;
    most = 0;
    for (int v = 0; v < n_values; ++v) {
        if (src[v] == nullptr || dst[v] == nullptr) ASH_FAIL("null value tensor");
        if (row_bytes[v] <= 0 || row_bytes[v] % 4 != 0) {
            ASH_FAIL("gather_rows: rows must be a positive multiple of 4 bytes");
        }
        if (src_rows[v] < 0) ASH_FAIL("negative source row count");
        a.src[v] = static_cast<const uint32_t*>(src[v]);
        a.dst[v] = static_cast<uint32_t*>(dst[v]);
        a.row_dwords[v] = static_cast<int32_t>(row_bytes[v] / 4);
        a.src_rows[v] = src_rows[v];
        most = std::max(most, n * a.row_dwords[v]);
    }
    return 0;
}

// Rounds of 1024 indices that a workgroup of a listing takes: eight where one
// workgroup then takes them all (and lists them in order); else one while that makes
// no more workgroups than there are CUs, so that a small table keeps the device busy;
// more beyond, where the updates of the cursor would queue.  (Rows of 16 bytes along,
// us with 1 / 4 / 8: 500 000 indices 12.3 / 10.9 / 14.9, 1.6 M 26.9 / 18.6 / 20.0, 24 M
// - / 235 / 240; keys alone 1.6 M - / 10.9 / 10.6, 24 M - / 103 / 98.)
int items_rounds(int64_t capacity, bool rows) {
    if (capacity <= 8 * kItemsBlock) return 8;
    if (capacity <= 256 * kItemsBlock) return 1;
    return rows || capacity <= 1024 * kItemsBlock ? 4 : 8;
}

template <int DIM>
void launch_items(const ash_map* map, int32_t* keys_out, int64_t* indices_out, int64_t n, int identity,
                  const GatherArgs& rows, int slot, bool last, hipStream_t s) {
    const int rounds = items_rounds(map->capacity, rows.n > 0);
    auto kernel = rounds == 1   ? items_kernel<DIM, 1>
                  : rounds == 4 ? items_kernel<DIM, 4>
                                : items_kernel<DIM, 8>;
    kernel<<<grid_for(map->capacity, kItemsBlock * rounds), kItemsBlock, 0, s>>>(
            map->d, keys_out, indices_out, n, identity, rows, slot, last);
}

}  // namespace

// Every entry that reads or updates buckets calls this first.  The fill must
// not end up in a captured graph: replays would empty the table again.
int settle_table(ash_map* map, hipStream_t s) {
    if (!map->table_stale) return 0;
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &capturing) == hipSuccess &&
        capturing != hipStreamCaptureStatusNone) {
        ASH_FAIL("the table was cleared and not used since: run one call outside the capture first");
    }
    if (map->table_filled) {
        map->table_stale = map->table_filled = false;
        return 0;
    }
    return fill_buckets(map, s);
}

Change::Change(ash_map* map, ChangeKind kind, hipStream_t s) : map_(map) {
    if (kind != kChangeElse && is_capturing(s)) map->replayed = true;
    std::lock_guard<std::mutex> lock(map->counter_lock);
    map->changed_on = s;
    lapse();
    if (kind == kChangeAdds) ++map->unread_inserts;
    if (kind == kChangeErases) map->maybe_tombstones = true;
}

void Change::queued() {
    if (map_ == nullptr) return;
    std::lock_guard<std::mutex> lock(map_->counter_lock);
    lapse();
    map_ = nullptr;
}

void Change::queued_with(const ash_counters& c) {
    std::lock_guard<std::mutex> lock(map_->counter_lock);
    lapse();
    map_->counters = c;
    map_->counters_known = true;
    map_ = nullptr;
}

void Change::lapse() {
    ++map_->changes;
    map_->counters_known = false;
    map_->late_pending = false;   // what a queued read-back brings is out of date
}

int check_batch(const ash_map* map, const void* keys, int64_t n) {
    if (check_map(map)) return 1;
    if (n < 0) ASH_FAIL("negative key count");
    if (n > 0 && keys == nullptr) ASH_FAIL("null keys pointer");
    if (n > (int64_t{1} << 31) - kHeapBlock) ASH_FAIL("too many keys in one call");
    return 0;
}

int check_rows(int n_values, const void* const* src, void* const* dst, const int64_t* row_bytes) {
    if (n_values < 0) ASH_FAIL("negative value count");
    if (n_values > 0 && (src == nullptr || dst == nullptr || row_bytes == nullptr)) {
        ASH_FAIL("null value tables");
    }
    for (int v = 0; v < n_values; ++v) {
        if (src[v] == nullptr || dst[v] == nullptr) ASH_FAIL("null value tensor");
        if (row_bytes[v] <= 0) ASH_FAIL("value rows must not be empty");
    }
    return 0;
}

int erase_selected(ash_map* map, bool codes, const void* keys, const int32_t* sel,
                   const int32_t* nsel, hipStream_t s) {
    const int32_t* k = static_cast<const int32_t*>(keys);
    constexpr unsigned g = 64;   // the selection is empty or short as a rule
    if (codes) {
        erase_selected_kernel<1, true><<<g, kEraseBlock, 0, s>>>(map->d, k, sel, nsel);
    } else {
        switch (map->key_dim) {
            case 1:
                erase_selected_kernel<1, false><<<g, kEraseBlock, 0, s>>>(map->d, k, sel, nsel);
                break;
            case 2:
                erase_selected_kernel<2, false><<<g, kEraseBlock, 0, s>>>(map->d, k, sel, nsel);
                break;
            case 3:
                erase_selected_kernel<3, false><<<g, kEraseBlock, 0, s>>>(map->d, k, sel, nsel);
                break;
            default:
                erase_selected_kernel<4, false><<<g, kEraseBlock, 0, s>>>(map->d, k, sel, nsel);
                break;
        }
    }
    ASH_LAUNCH_CHECK();
    return 0;
}

int insert_selected(ash_map* map, bool codes, const void* keys,
                    const int32_t* sel, const int32_t* nsel,
                    const ValueArgs& va, hipStream_t s, const Publish& publish) {
    const int32_t* k = static_cast<const int32_t*>(keys);
    if (va.n > 0) {
        return launch_selected<kInsertFused>(map, codes, k, sel, nsel, va, s, publish);
    }
    return launch_selected<kInsertKeys>(map, codes, k, sel, nsel, va, s, publish);
}

namespace {

// When the rows are read in index order, and what that takes.  Measured (key by
// key -> in index order, us; keys stored unless said otherwise):
//   two tables or more; of one (rows of 12 bytes) the passes cost what its lines do
//   2 M queries and more: rows of 12 + 4 bytes, 1.5 M rows: 1 M queries 46 -> 58,
//     2 M 90 -> 81, 4 M 183 -> 151, 8 M 374 -> 280
//   16 MB of tables: 6 MB (of which an XCD's L2 holds most) and 4 M queries 111 ->
//     123, 12 MB 200 -> 173
//   queries per row of the tables, of which fewer share no lines in a part: for rows
//     of up to 16 bytes together a quarter (400 MB of tables: 8 bytes 743 -> 610, 16
//     bytes 391 -> 359), for wider ones one (400 MB: a half 20 bytes 617 -> 583, 24
//     bytes 510 -> 513, 32 bytes 403 -> 427; one 1185 -> 1052, 1014 -> 948, 768 ->
//     774).  From 900 MB of tables on, where a random line costs a translation as
//     well, a quarter does for rows of up to 24 bytes (1 GB: 781 -> 706) and a half
//     for 32 (a quarter 572 -> 587, a half 1132 -> 1042).  Parts that an L2 does not
//     hold are no loss there: 3 GB, rows of 16 bytes 3747 -> 3079.
//   rows of up to kSortMaxWords words together: a chunk's have to fit the LDS.
// A key that is not stored costs key by key only the line of its bucket.  Pass 1 hence
// counts a chunk's stored keys, and below a share of them serves the chunk itself: of
// 8 bytes three eighths (400 MB, 25 M queries: four tenths stored 1036 -> 962, three
// 946 -> 1027), of 16 a half (seven tenths 623 -> 591, a half 536 -> 551), of wider
// ones seven eighths, six from 900 MB on.  What is left of the passes costs such a
// chunk 2 - 12 % over key by key while three tenths of its keys are stored (22 % where
// the call takes 0.1 - 0.2 ms) and up to 30 % (a tenth of a millisecond at 25 M) where
// next to none is; through all three passes that was 45 %.
// (Looking at a chunk's first 512 keys and then going key by key at once: the
// registers of both ways together cost 10 - 40 %.)
constexpr int64_t kSortMinQueries = int64_t{1} << 21;
constexpr int64_t kSortMinBytes = int64_t{16} << 20;
constexpr int64_t kSortFarBytes = int64_t{900} << 20;

int64_t plan_row_sort(int64_t n, int n_values, const int64_t* row_bytes, const int64_t* src_rows,
                      void* scratch, RowSort* sort) {
    if (n < kSortMinQueries || n > 0x7FFF0000ll || n_values < 2 || n_values > kMaxFusedValues) return 0;
    int64_t words = 0, rows = 0, table_bytes = 0;
    for (int v = 0; v < n_values; ++v) {
        if (row_bytes[v] <= 0 || row_bytes[v] % 4 != 0 || src_rows[v] < 0 || src_rows[v] > 0x7FFFFFFFll) return 0;
        if (row_bytes[v] > 4 * kSortMaxWords) return 0;
        words += row_bytes[v] / 4;
        rows = std::max(rows, src_rows[v]);
        table_bytes += row_bytes[v] * src_rows[v];
    }
    if (words > kSortMaxWords || rows <= kSortParts || table_bytes < kSortMinBytes) return 0;
    const bool far = table_bytes >= kSortFarBytes;
    if (n < (words <= 4 || (far && words <= 6) ? rows / 4 : far ? rows / 2 : rows)) return 0;
    const int64_t chunks = (n + kSortChunk - 1) / kSortChunk;
    int64_t off = 0;
    auto take = [&](int64_t bytes) {
        char* p = scratch != nullptr ? static_cast<char*>(scratch) + off : nullptr;
        off += (bytes + 255) & ~int64_t{255};
        return p;
    };
    void* index = take(chunks * kSortChunk * 4);
    void* place = take(n * 2);
    void* bounds = take(chunks * kSortBounds * 2);
    void* out = take(chunks * kSortChunk * words * 4);
    if (sort != nullptr) {
        *sort = {n, static_cast<uint32_t>(chunks),
                 static_cast<uint32_t>((static_cast<uint64_t>(kSortParts) << 32) / static_cast<uint64_t>(rows)),
                 static_cast<uint32_t>(words), words <= 2 ? 3 : words <= 4 ? 4 : far ? 6 : 7,
                 static_cast<int32_t*>(index), static_cast<uint16_t*>(place),
                 static_cast<uint16_t*>(bounds), static_cast<uint32_t*>(out)};
    }
    return off;
}

int find_rows_sorted(ash_map* map, const int32_t* keys, RowTables tabs, const RowSort& sort, int miss,
                     int64_t* indices, uint8_t* masks, hipStream_t s) {
    switch (map->key_dim) {
        case 1: find_sort_kernel<1><<<sort.chunks, kSortThreads, 0, s>>>(map->d, keys, sort, tabs, miss, indices, masks); break;
        case 2: find_sort_kernel<2><<<sort.chunks, kSortThreads, 0, s>>>(map->d, keys, sort, tabs, miss, indices, masks); break;
        case 3: find_sort_kernel<3><<<sort.chunks, kSortThreads, 0, s>>>(map->d, keys, sort, tabs, miss, indices, masks); break;
        default: find_sort_kernel<4><<<sort.chunks, kSortThreads, 0, s>>>(map->d, keys, sort, tabs, miss, indices, masks); break;
    }
    ASH_LAUNCH_CHECK();
    // these two address rows by words
    for (int v = 0; v < tabs.n; ++v) {
        if ((tabs.wide >> v) & 1u) tabs.units[v] *= 4;
        tabs.magic[v] = static_cast<uint32_t>((0x100000000ull + tabs.units[v] - 1) / tabs.units[v]);
    }
    tabs.wide = 0;
    constexpr uint32_t kRunsPerGroup = kSortRuns * (kBlock / 64);
    const uint32_t groups = (sort.chunks + kRunsPerGroup - 1) / kRunsPerGroup;
    const unsigned g = groups * kSortParts;
    switch (sort.words) {
        case 2: gather_parts_kernel<2><<<g, kBlock, 0, s>>>(tabs, sort, groups); break;
        case 3: gather_parts_kernel<3><<<g, kBlock, 0, s>>>(tabs, sort, groups); break;
        case 4: gather_parts_kernel<4><<<g, kBlock, 0, s>>>(tabs, sort, groups); break;
        case 5: gather_parts_kernel<5><<<g, kBlock, 0, s>>>(tabs, sort, groups); break;
        case 6: gather_parts_kernel<6><<<g, kBlock, 0, s>>>(tabs, sort, groups); break;
        case 7: gather_parts_kernel<7><<<g, kBlock, 0, s>>>(tabs, sort, groups); break;
        default: gather_parts_kernel<8><<<g, kBlock, 0, s>>>(tabs, sort, groups); break;
    }
    ASH_LAUNCH_CHECK();
    const size_t lds = static_cast<size_t>(kSortChunk) * (sort.words * 4 + 2);
    ASH_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(deal_rows_kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
    deal_rows_kernel<<<sort.chunks, kDealThreads, lds, s>>>(tabs, sort, miss);
    ASH_LAUNCH_CHECK();
    return 0;
}

}  // namespace

}  // namespace ash

using namespace ash;

extern "C" {

const char* ash_last_error(void) { return g_last_error.c_str(); }

int ash_abi_version(void) { return 1; }

// The build passes the fingerprint of the kernel sources it compiles
// (torch-ash_amd/build.py: source_fingerprint).
#ifndef ASH_SOURCE_FINGERPRINT
#define ASH_SOURCE_FINGERPRINT "unknown"
#endif
const char* ash_source_fingerprint(void) { return ASH_SOURCE_FINGERPRINT; }

int ash_map_workspace_bytes(int key_dim, int64_t capacity, int64_t* table_bytes,
                            int64_t* general_bytes) {
    if (key_dim < 1 || key_dim > 4) ASH_FAIL("key_dim must be in 1..4");
    if (capacity < 1 || capacity > 0x7FFFFFF0ll) {
        ASH_FAIL("capacity must be in 1..2^31-16");
    }
    if (table_bytes) *table_bytes = table_workspace_bytes(capacity);
    if (general_bytes) *general_bytes = general_slots(capacity) * 20;
    return 0;
}

int ash_map_create(int key_dim, int64_t capacity, int32_t* heap, void* table_ws,
                   int64_t table_bytes, int device, void* stream,
                   ash_map_t** out) {
    if (out == nullptr) ASH_FAIL("null output handle");
    *out = nullptr;
    int64_t need = 0;
    if (ash_map_workspace_bytes(key_dim, capacity, &need, nullptr)) return 1;
    if (heap == nullptr || table_ws == nullptr) ASH_FAIL("null device buffer");
    if (table_bytes < need) ASH_FAIL("table workspace too small");
    if (reinterpret_cast<uintptr_t>(table_ws) % 256 != 0) {
        ASH_FAIL("table workspace must be 256-byte aligned");
    }
    DeviceGuard guard;
    ASH_HIP(guard.enter(device));
    ash_map* map = new ash_map();
    map->key_dim = key_dim;
    map->capacity = capacity;
    map->device = device;
    map->table_bytes = table_bytes;
    map->general_attached = false;
    map->table_stale = map->table_filled = false;
    map->heap_dirty = true;   // the caller's buffer holds anything
    map->log_stale = false;
    map->line = nullptr;
    map->stamp = map->late_stamp = 0;
    map->late_in_flight = map->late_pending = map->late_of_erase = false;
    map->counters_known = true;   // a new map is empty and every counter is zero
    map->counters = {};
    map->maybe_tombstones = false;
    map->unread_inserts = 0;
    map->launches = 0;
    map->changes = 0;
    map->changed_on = static_cast<hipStream_t>(stream);
    map->replayed = false;
    map->d.ctr = static_cast<int32_t*>(table_ws);
    map->d.buckets = reinterpret_cast<uint64_t*>(static_cast<char*>(table_ws) +
                                                 kHeaderBytes);
    map->d.klog = reinterpret_cast<uint64_t*>(static_cast<char*>(table_ws) +
                                              klog_offset(capacity));
    map->d.heap = heap;
    map->d.gstate = nullptr;
    map->d.gkeys = nullptr;
    map->d.nb = static_cast<uint32_t>(num_buckets(capacity));
    map->d.gslots = 0;
    map->d.capacity = static_cast<int32_t>(capacity);
    if (clear_lazily(map, static_cast<hipStream_t>(stream), true, {})) {
        delete map;
        return 1;
    }
    *out = map;
    return 0;
}

int ash_map_attach_general(ash_map_t* map, void* general_ws,
                           int64_t general_bytes, void* stream) {
    if (check_map(map)) return 1;
    if (map->general_attached) ASH_FAIL("general region already attached");
    if (general_ws == nullptr || general_bytes < kMinGeneralSlots * 20) {
        ASH_FAIL("general workspace too small");
    }
    // the largest power of two of slots that fits, up to what `capacity` keys need
    int64_t slots = kMinGeneralSlots;
    while (slots < general_slots(map->capacity) && slots * 2 * 20 <= general_bytes) slots <<= 1;
    if (reinterpret_cast<uintptr_t>(general_ws) % 256 != 0) {
        ASH_FAIL("general workspace must be 256-byte aligned");
    }
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    // (what an insert before leaves for the host is not lost)
    ash_counters before;
    bool known;
    {
        std::lock_guard<std::mutex> lock(map->counter_lock);
        if (take_late_words(map)) return 1;
        before = map->counters;
        known = map->counters_known;
    }
    Change change(map, kChangeElse, s);
    // keys first (16 B per slot, keeps them 16-byte aligned), then states
    map->d.gkeys = static_cast<int32_t*>(general_ws);
    map->d.gstate = map->d.gkeys + slots * 4;
    map->d.gslots = static_cast<uint32_t>(slots);
    map->general_attached = true;
    fill16_kernel<<<capped_grid(slots / 4), kBlock, 0, s>>>(
            reinterpret_cast<uint4*>(map->d.gstate), slots / 4, 0xFFFFFFFFu);
    ASH_LAUNCH_CHECK();
    set_counter_kernel<<<1, 64, 0, s>>>(map->d.ctr, kCtrExotic, 0);
    ASH_LAUNCH_CHECK();
    before.exotic_pending = 0;
    if (known) change.queued_with(before);
    return 0;
}

int ash_map_destroy(ash_map_t* map) {
    if (map == nullptr) return 0;
    // words that the device may still owe must have arrived before their line
    // serves another map or call
    if (map->late_in_flight) {
        DeviceGuard guard;
        (void)guard.enter(map->device);
        std::lock_guard<std::mutex> lock(map->counter_lock);
        (void)settle_late_words(map);
    }
    if (!map->late_in_flight) give_back_line(map->line);
    delete map;
    return 0;
}

int ash_map_find(ash_map_t* map, const int32_t* keys, int64_t n,
                 int64_t* indices, uint8_t* masks, void* stream) {
    if (check_batch(map, keys, n)) return 1;
    if (n == 0) return 0;
    if (indices == nullptr || masks == nullptr) ASH_FAIL("null output pointer");
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (settle_table(map, s)) return 1;
    const unsigned g = grid_for(n);
    auto launch = [&](auto dim) {
        constexpr int DIM = decltype(dim)::value;
        const auto kernel = n <= kAloneKeys ? find_kernel<DIM, true> : find_kernel<DIM, false>;
        kernel<<<g, kBlock, 0, s>>>(map->d, keys, n, indices, masks);
    };
    switch (map->key_dim) {
        case 1: launch(std::integral_constant<int, 1>{}); break;
        case 2: launch(std::integral_constant<int, 2>{}); break;
        case 3: launch(std::integral_constant<int, 3>{}); break;
        default: launch(std::integral_constant<int, 4>{}); break;
    }
    ASH_LAUNCH_CHECK();
    return 0;
}

int ash_map_find_rows(ash_map_t* map, const int32_t* keys, int64_t n, int n_values,
                      const void* const* src, void* const* dst, const int64_t* row_bytes,
                      const int64_t* src_rows, int zero_misses, int64_t* indices,
                      uint8_t* masks, void* stream) {
    return ash_map_find_rows_scratch(map, keys, n, n_values, src, dst, row_bytes, src_rows, zero_misses,
                                     indices, masks, nullptr, 0, stream);
}

int64_t ash_map_find_rows_scratch_bytes(const ash_map_t* map, int64_t n, int n_values,
                                        const int64_t* row_bytes, const int64_t* src_rows) {
    if (map == nullptr || row_bytes == nullptr || src_rows == nullptr) return 0;
    return plan_row_sort(n, n_values, row_bytes, src_rows, nullptr, nullptr);
}

int ash_map_find_rows_scratch(ash_map_t* map, const int32_t* keys, int64_t n, int n_values,
                              const void* const* src, void* const* dst, const int64_t* row_bytes,
                              const int64_t* src_rows, int zero_misses, int64_t* indices,
                              uint8_t* masks, void* scratch, int64_t scratch_bytes, void* stream) {
    if (check_batch(map, keys, n)) return 1;
    if (n_values < 0 || n_values > kMaxFusedValues) {
        ASH_FAIL("find_rows takes up to " + std::to_string(kMaxFusedValues) + " tensors per call");
    }
    if (n_values > 0 && (src == nullptr || dst == nullptr || row_bytes == nullptr || src_rows == nullptr)) {
        ASH_FAIL("null value tables");
    }
    RowTables tabs = {};
    tabs.n = n_values;
    for (int v = 0; v < n_values; ++v) {
        if (n > 0 && (src[v] == nullptr || dst[v] == nullptr)) ASH_FAIL("null value tensor");
        if (row_bytes[v] <= 0 || row_bytes[v] % 4 != 0) {
            ASH_FAIL("find_rows: rows must be a positive multiple of 4 bytes");
        }
        if (src_rows[v] < 0 || src_rows[v] > 0x7FFFFFFFll) ASH_FAIL("find_rows: bad source row count");
        const bool wide = (reinterpret_cast<uintptr_t>(src[v]) | reinterpret_cast<uintptr_t>(dst[v]) |
                           static_cast<uintptr_t>(row_bytes[v])) % 16 == 0;
        const int64_t units = row_bytes[v] / (wide ? 16 : 4);
        if (units > kMaxRowUnits) ASH_FAIL("find_rows: rows of at most 32764 bytes");
        if (wide) tabs.wide |= 1u << v;
        tabs.src[v] = src[v];
        tabs.dst[v] = dst[v];
        tabs.units[v] = static_cast<uint32_t>(units);
        tabs.magic[v] = static_cast<uint32_t>((0x100000000ull + units - 1) / units);
        tabs.src_rows[v] = static_cast<uint32_t>(src_rows[v]);
    }
    if (n == 0) return 0;
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (settle_table(map, s)) return 1;
    const int miss = zero_misses ? -1 : 0;
    if (scratch != nullptr && reinterpret_cast<uintptr_t>(scratch) % 16 == 0) {
        RowSort sort;
        const int64_t need = plan_row_sort(n, n_values, row_bytes, src_rows, scratch, &sort);
        if (need > 0 && scratch_bytes >= need) {
            return find_rows_sorted(map, keys, tabs, sort, miss, indices, masks, s);
        }
    }
    const unsigned g = grid_for(n);
    auto launch = [&](auto dim) {
        constexpr int DIM = decltype(dim)::value;
        const auto kernel = n <= kAloneKeysWithRows ? find_rows_kernel<DIM, true> : find_rows_kernel<DIM, false>;
        kernel<<<g, kBlock, 0, s>>>(map->d, keys, n, tabs, miss, indices, masks);
    };
    switch (map->key_dim) {
        case 1: launch(std::integral_constant<int, 1>{}); break;
        case 2: launch(std::integral_constant<int, 2>{}); break;
        case 3: launch(std::integral_constant<int, 3>{}); break;
        default: launch(std::integral_constant<int, 4>{}); break;
    }
    ASH_LAUNCH_CHECK();
    return 0;
}

int ash_add_rows(const void* rows, const int64_t* indices, const uint8_t* masks, int64_t n,
                 int64_t width, int dtype, void* out, int64_t out_rows, void* stream) {
    if (n < 0 || width < 1 || out_rows < 0) ASH_FAIL("add_rows: bad sizes");
    if (dtype != ASH_F32 && dtype != ASH_F64) ASH_FAIL("add_rows: dtype must be float32 or float64");
    if (out == nullptr && out_rows > 0) ASH_FAIL("null output pointer");
    if (n > 0 && (rows == nullptr || indices == nullptr || masks == nullptr)) {
        ASH_FAIL("null pointer in add_rows");
    }
    if (out_rows == 0) return 0;
    if (reinterpret_cast<uintptr_t>(out) % 16 != 0) ASH_FAIL("add_rows: the output must be 16-byte aligned");
    PointerGuard guard;
    ASH_HIP(guard.enter_for(out));
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t bytes = out_rows * width * (dtype == ASH_F32 ? 4 : 8);
    clear_rows_kernel<<<capped_grid((bytes + 15) / 16), kBlock, 0, s>>>(static_cast<uint32_t*>(out),
                                                                       bytes / 4);
    ASH_LAUNCH_CHECK();
    if (n == 0) return 0;
    const unsigned g = capped_grid(n * width);
    if (dtype == ASH_F32) {
        add_rows_kernel<float><<<g, kBlock, 0, s>>>(static_cast<const float*>(rows), indices, masks, n,
                                                    width, static_cast<float*>(out), out_rows);
    } else {
        add_rows_kernel<double><<<g, kBlock, 0, s>>>(static_cast<const double*>(rows), indices, masks, n,
                                                     width, static_cast<double*>(out), out_rows);
    }
    ASH_LAUNCH_CHECK();
    return 0;
}

int ash_grid_query(ash_map_t* map, const float* x, int64_t n, int grid_dim,
                   int64_t* grid_indices, int64_t* cell_indices, float* offsets,
                   uint8_t* masks, void* stream) {
    if (check_batch(map, x, n)) return 1;
    if (map->key_dim != 3) ASH_FAIL("grid queries need a map with 3-d keys");
    if (grid_dim < 1 || grid_dim > 1024) ASH_FAIL("grid_dim must be in 1..1024");
    if (n == 0) return 0;
    if (grid_indices == nullptr || cell_indices == nullptr ||
        offsets == nullptr || masks == nullptr) {
        ASH_FAIL("null output pointer");
    }
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    if (settle_table(map, static_cast<hipStream_t>(stream))) return 1;
    grid_query_kernel<<<grid_for(n), kBlock, 0,
                        static_cast<hipStream_t>(stream)>>>(
            map->d, x, n, static_cast<float>(grid_dim), grid_dim, grid_indices,
            cell_indices, offsets, masks);
    ASH_LAUNCH_CHECK();
    return 0;
}

namespace {

// Argument checks shared by the two activation entry points; `heads` is
// checked by the caller.
int check_activate(ash_map_t* map, const float* cells, int64_t n, int grid_dim,
                   int dilation, int bound_lo, int bound_hi, const uint8_t* touched,
                   const int32_t* coords) {
    if (check_batch(map, cells, n)) return 1;
    if (map->key_dim != 3) ASH_FAIL("block activation needs a map with 3-d keys");
    if (grid_dim < 1 || grid_dim > 1024) ASH_FAIL("grid_dim must be in 1..1024");
    if (dilation < 0 || dilation > 8) ASH_FAIL("dilation must be in 0..8");
    if (bound_lo > bound_hi) ASH_FAIL("empty block bounds");
    if (n > 0 && (touched == nullptr || coords == nullptr)) {
        ASH_FAIL("null output or scratch pointer");
    }
    return 0;
}

// The launches of an activation; the map's device is current, `heads` points
// to 64 + 3 n int32 of device memory.
int launch_activate(ash_map_t* map, const float* cells, int64_t n, int grid_dim,
                    int dilation, int bidirectional, int bound_lo, int bound_hi,
                    uint8_t* touched, int32_t* coords, int32_t* heads, hipStream_t s) {
    if (settle_table(map, s)) return 1;
    Change change(map, kChangeAdds, s);
    const int lo = bidirectional ? -dilation : 0;
    const int width = dilation - lo + 1;
    const float g = static_cast<float>(grid_dim);
    set_counter_kernel<<<1, 64, 0, s>>>(heads, 0, 0);
    ASH_LAUNCH_CHECK();
    activate_heads_kernel<<<grid_for(n, kHeadsBlock), kHeadsBlock, 0, s>>>(
            cells, n, g, bound_lo, bound_hi, heads);
    ASH_LAUNCH_CHECK();
    int64_t blocks = (n * width * width * width + kHeapBlock - 1) / kHeapBlock;
    if (blocks > 2048) blocks = 2048;
    const unsigned gb = static_cast<unsigned>(blocks);
    auto insert = tombs_in(map) ? activate_kernel<false, true> : activate_kernel<false, false>;
    insert<<<gb, kHeapBlock, 0, s>>>(
            map->d, heads, lo, width, bound_lo, bound_hi, touched, coords);
    ASH_LAUNCH_CHECK();
    activate_kernel<true, false><<<gb, kHeapBlock, 0, s>>>(
            map->d, heads, lo, width, bound_lo, bound_hi, touched, coords);
    ASH_LAUNCH_CHECK();
    return 0;
}

// Address of `scratch` on each device, asked for once per device with that
// device current (every device holds its own copy at its own address).
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
int32_t* g_scratch_ptr[kMaxDevices] = {};

int scratch_on_current_device(int device, int32_t** out) {
    if (device < 0 || device >= kMaxDevices) ASH_FAIL("device number out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[device] == nullptr) {
        void* p = nullptr;
        ASH_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (p == nullptr) ASH_FAIL("hipGetSymbolAddress returned no address for the scratch array");
        g_scratch_ptr[device] = static_cast<int32_t*>(p);
    }
    *out = g_scratch_ptr[device];
    return 0;
}

}  // namespace

int ash_grid_activate(ash_map_t* map, const float* cells, int64_t n,
                      int grid_dim, int dilation, int bidirectional,
                      int bound_lo, int bound_hi, uint8_t* touched,
                      int32_t* coords, int32_t* heads_scratch, void* stream) {
    if (check_activate(map, cells, n, grid_dim, dilation, bound_lo, bound_hi, touched, coords)) {
        return 1;
    }
    if (n == 0) return 0;
    if (heads_scratch == nullptr) ASH_FAIL("null output or scratch pointer");
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    return launch_activate(map, cells, n, grid_dim, dilation, bidirectional, bound_lo, bound_hi,
                           touched, coords, heads_scratch, static_cast<hipStream_t>(stream));
}

int ash_grid_activate_static(ash_map_t* map, const float* cells, int64_t n,
                             int grid_dim, int dilation, int bidirectional,
                             int bound_lo, int bound_hi, uint8_t* touched,
                             int32_t* coords, void* stream) {
    if (check_activate(map, cells, n, grid_dim, dilation, bound_lo, bound_hi, touched, coords)) {
        return 1;
    }
    if (n > kActivateStaticMax) {
        ASH_FAIL("ash_grid_activate_static takes at most " +
                 std::to_string(kActivateStaticMax) +
                 " positions per call (ASH_ACTIVATE_STATIC_MAX_POSITIONS); use "
                 "ash_grid_activate with a scratch buffer of the caller's for more");
    }
    if (n == 0) return 0;
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    int32_t* heads = nullptr;
    if (scratch_on_current_device(map->device, &heads)) return 1;
    return launch_activate(map, cells, n, grid_dim, dilation, bidirectional, bound_lo, bound_hi,
                           touched, coords, heads, static_cast<hipStream_t>(stream));
}

int ash_grid_activate_positions(ash_map_t* map, const float* positions, int64_t n,
                                const float* origin, float cell_size, int grid_dim,
                                int dilation, int bidirectional, int bound_lo, int bound_hi,
                                uint8_t* touched, int32_t* coords, void* stream) {
    if (check_activate(map, positions, n, grid_dim, dilation, bound_lo, bound_hi, touched,
                       coords)) {
        return 1;
    }
    if (!(cell_size > 0.f) || !(cell_size < INFINITY)) ASH_FAIL("cell_size must be positive and finite");
    if (n == 0) return 0;
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool empty = map->table_stale;
    if (settle_table(map, s)) return 1;
    Change change(map, kChangeAdds, s);
    RunsArgs a;
    a.x = positions;
    a.origin = origin;
    a.inv_cell = 1.0f / cell_size;
    a.g = static_cast<float>(grid_dim);
    a.n = n;
    a.off_lo = bidirectional ? -dilation : 0;
    a.width = dilation - a.off_lo + 1;
    a.bound_lo = bound_lo;
    a.bound_hi = bound_hi;
    a.empty = empty;
    const int64_t groups = (n + kRunPositions - 1) / kRunPositions;
    if (groups > 0x7FFFFFFFll) ASH_FAIL("too many positions in one call");
    const bool alone = !empty || groups <= 2 * compute_units();
    auto kernel = tombs_in(map) ? (alone ? activate_runs_kernel<true, true> : activate_runs_kernel<true, false>)
                                : (alone ? activate_runs_kernel<false, true> : activate_runs_kernel<false, false>);
    kernel<<<static_cast<unsigned>(groups), kHeapBlock, 0, s>>>(map->d, a, touched, coords);
    ASH_LAUNCH_CHECK();
    return 0;
}

namespace {
int insert_per_key(ash_map* map, const int32_t* keys, int64_t n, int n_values,
                   const void* const* src, void* const* dst, const int64_t* row_bytes,
                   int32_t* assigned, void* stream, const Publish& publish = {}, const KeyCheck& check = {});
}

int ash_map_insert_keys(ash_map_t* map, const int32_t* keys, int64_t n,
                        void* stream) {
    return insert_per_key(map, keys, n, 0, nullptr, nullptr, nullptr, nullptr, stream);
}

int ash_map_insert_needs_scratch(int n_values, const int64_t* row_bytes) {
    if (n_values <= 0) return 0;
    if (n_values > kMaxFusedValues) return 1;
    for (int v = 0; v < n_values; ++v) {
        if (row_bytes[v] % 4 != 0 || row_bytes[v] > kMaxFusedRowDwords * 4) {
            return 1;
        }
    }
    return 0;
}

int ash_scatter_rows(const void* src, void* dst, const int32_t* assigned,
                     int64_t n, int64_t row_bytes, void* stream) {
    if (n == 0 || row_bytes == 0) return 0;
    if (src == nullptr || dst == nullptr || assigned == nullptr) {
        ASH_FAIL("null pointer in scatter");
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const uintptr_t align = reinterpret_cast<uintptr_t>(src) |
                            reinterpret_cast<uintptr_t>(dst) |
                            static_cast<uintptr_t>(row_bytes);
    if (align % 16 == 0) {
        const int64_t upr = row_bytes / 16;
        scatter_rows_kernel<uint4><<<looping_grid(n * upr), kBlock, 0, s>>>(
                static_cast<const uint4*>(src), static_cast<uint4*>(dst),
                assigned, n, upr);
    } else if (align % 4 == 0) {
        const int64_t upr = row_bytes / 4;
        scatter_rows_kernel<uint32_t><<<looping_grid(n * upr), kBlock, 0, s>>>(
                static_cast<const uint32_t*>(src), static_cast<uint32_t*>(dst),
                assigned, n, upr);
    } else {
        scatter_rows_kernel<uint8_t><<<looping_grid(n * row_bytes), kBlock, 0,
                                       s>>>(static_cast<const uint8_t*>(src),
                                            static_cast<uint8_t*>(dst),
                                            assigned, n, row_bytes);
    }
    ASH_LAUNCH_CHECK();
    return 0;
}

int ash_gather_rows(int n_values, const void* const* src, void* const* dst,
                    const int64_t* row_bytes, const int64_t* src_rows,
                    const int64_t* indices, int64_t n, void* stream) {
    if (n_values < 1 || n_values > kMaxFusedValues) {
        ASH_FAIL("gather_rows takes 1.." + std::to_string(kMaxFusedValues) + " tensors per call");
    }
    if (n < 0) ASH_FAIL("negative row count");
    GatherArgs a;
    int64_t most = 0;
    if (n > 0 && gather_args(n_values, src, dst, row_bytes, src_rows, n, a, most)) return 1;
    if (n == 0 && (src == nullptr || dst == nullptr || row_bytes == nullptr || src_rows == nullptr)) {
        ASH_FAIL("null value tables");
    }
    if (n == 0) return 0;
    PointerGuard guard;
    ASH_HIP(guard.enter_for(src[0]));
    if (indices == nullptr) {
        int64_t g = (most / 4 + kBlock - 1) / kBlock;
        if (g > 256 * 64) g = 256 * 64;
        if (g < 1) g = 1;
        copy_first_rows_kernel<<<static_cast<unsigned>(g), kBlock, 0,
                                 static_cast<hipStream_t>(stream)>>>(a, n);
        ASH_LAUNCH_CHECK();
        return 0;
    }
    gather_rows_kernel<<<looping_grid(most), kBlock, 0, static_cast<hipStream_t>(stream)>>>(
            a, indices, n);
    ASH_LAUNCH_CHECK();
    return 0;
}

namespace {

// `publish`: what the launch that changes the counters leaves for the host.
int insert_per_key(ash_map* map, const int32_t* keys, int64_t n, int n_values,
                   const void* const* src, void* const* dst, const int64_t* row_bytes,
                   int32_t* assigned, void* stream, const Publish& publish,
                   const KeyCheck& check) {
    if (check_batch(map, keys, n) || check_rows(n_values, src, dst, row_bytes)) return 1;
    if (n == 0) return 0;
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (settle_table(map, s)) return 1;
    Change change(map, kChangeAdds, s);
    ValueArgs va = {};
    if (n_values == 0) return launch_insert<kInsertKeys>(map, keys, n, va, nullptr, nullptr, s, publish, check);
    if (!ash_map_insert_needs_scratch(n_values, row_bytes)) {
        va.n = n_values;
        for (int v = 0; v < n_values; ++v) {
            va.src[v] = static_cast<const uint32_t*>(src[v]);
            va.dst[v] = static_cast<uint32_t*>(dst[v]);
            va.row_dwords[v] = static_cast<int32_t>(row_bytes[v] / 4);
        }
        return launch_insert<kInsertFused>(map, keys, n, va, nullptr, nullptr, s, publish, check);
    }
    if (assigned == nullptr) {
        ASH_FAIL("these value rows need the `assigned` temporary");
    }
    if (launch_insert<kInsertAssign>(map, keys, n, va, assigned, nullptr, s, publish, check)) {
        return 1;
    }
    for (int v = 0; v < n_values; ++v) {
        if (ash_scatter_rows(src[v], dst[v], assigned, n, row_bytes[v], stream)) {
            return 1;
        }
    }
    return 0;
}

}  // namespace

int ash_map_insert(ash_map_t* map, const int32_t* keys, int64_t n, int n_values,
                   const void* const* src, void* const* dst,
                   const int64_t* row_bytes, int32_t* assigned, void* stream) {
    return insert_per_key(map, keys, n, n_values, src, dst, row_bytes, assigned, stream);
}

int ash_map_erase(ash_map_t* map, const int32_t* keys, int64_t n,
                  void* stream) {
    if (check_batch(map, keys, n)) return 1;
    if (n == 0) return 0;
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (settle_table(map, s)) return 1;
    if (give_up_heap_order(map, s)) return 1;   // freed indices go back onto the heap
    Change change(map, kChangeErases, s);
    // Nobody waits here; but a size, a listing or an insert that follows wants the
    // counters, and finds them with a launch less.  (Not where the words of an
    // earlier call are still owed: a run of erases is not to wait for each other.)
    Publish publish = {};
    LatePlace late(map);
    if (n <= kLeaveKeys && !map->replayed && !is_capturing(s)) {
        if (late.take(false)) return 1;
        if (late.taken()) publish = {late.late(), late.stamp, next_ticket(map)};
    }
    auto launch = [&](auto block) {
        constexpr int BLOCK = decltype(block)::value;
        auto kernel = map->key_dim == 1   ? erase_kernel<1, BLOCK>
                      : map->key_dim == 2 ? erase_kernel<2, BLOCK>
                      : map->key_dim == 3 ? erase_kernel<3, BLOCK>
                                          : erase_kernel<4, BLOCK>;
        kernel<<<grid_for(n, BLOCK), BLOCK, 0, s>>>(map->d, keys, n, publish);
    };
    if (n <= kEraseBy256) launch(std::integral_constant<int, 256>{});
    else if (n <= kEraseBy512) launch(std::integral_constant<int, 512>{});
    else launch(std::integral_constant<int, kEraseBlock>{});
    ASH_LAUNCH_CHECK();
    change.queued();
    if (late.taken()) late.queued(true);
    return 0;
}

int ash_map_clear(ash_map_t* map, void* stream) {
    return ash_map_clear_rows(map, 0, nullptr, nullptr, stream);
}

int ash_map_clear_rows(ash_map_t* map, int n_values, void* const* rows, const int64_t* row_bytes,
                       void* stream) {
    if (check_map(map)) return 1;
    if (n_values < 0 || n_values > kMaxFusedValues) ASH_FAIL("clear: up to 4 value tables per call");
    if (n_values > 0 && (rows == nullptr || row_bytes == nullptr)) ASH_FAIL("null value tables");
    for (int v = 0; v < n_values; ++v) {
        if (row_bytes[v] < 0) ASH_FAIL("clear: negative size");
        if (row_bytes[v] > 0 && rows[v] == nullptr) ASH_FAIL("null value tensor");
        if (reinterpret_cast<uintptr_t>(rows[v]) % 16 != 0) ASH_FAIL("clear: values must be 16-byte aligned");
    }
    const ClearRows values = {n_values, rows, row_bytes};
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (is_capturing(s)) map->replayed = true;
    Change change(map, kChangeElse, s);
    if (map->replayed) {
        // what replays leave behind is unknown: everything is cleared now
        if (settle_table(map, s)) return 1;
        map->heap_dirty = true;
        if (clear_table(map, s, true, 0)) return 1;
        map->heap_dirty = true;   // (whatever the flag would say: see heap_in_order)
        ClearList list;
        list.add(values);
        if (list.launch(map, kCountersAsTheyAre, false, s)) return 1;
    } else if (clear_lazily(map, s, false, values)) {
        return 1;
    }
    // every counter is zero again: known without a read-back
    change.queued_with({});
    map->maybe_tombstones = false;
    map->unread_inserts = 0;
    return 0;
}

namespace {

// Who wants the counters: the call that changes the map, which is ordered behind all
// that have changed it; a reader, who may be another thread with a stream of its own;
// a reader who has the device asked in any case.
enum Asker { kOwnCall, kReader, kReaderOfDevice };

// The counters (the map's device is current): they are known already, or a read-back
// queued behind the latest insert brings them, or they are fetched now, which waits for
// `s`.  A reader of the device, too, asks behind words that are under way: they belong
// to a call that has returned.  What a reader has fetched is the latest state only if
// it was asked for on the stream of the latest change, behind that, and none has begun
// or been queued since; else it is the reader's alone.  (Replays change them on any
// stream: what is kept then holds for the call behind the reader's only.)
int refresh_counters(ash_map* map, hipStream_t s, Asker asker, ash_counters& c) {
    std::unique_lock<std::mutex> lock(map->counter_lock);
    if (map->replayed) {
        if (settle_late_words(map)) return 1;
        map->counters_known = map->late_pending = false;
    }
    if (take_late_words(map)) return 1;
    if (map->counters_known && asker != kReaderOfDevice) {
        c = map->counters;
        return 0;
    }
    if (is_capturing(s)) {
        ASH_FAIL("the table's counters cannot be read while the stream is being captured");
    }
    // (each of several readers waits for its own stream, not for the others)
    const uint32_t changes = map->changes;
    lock.unlock();
    Answer answer;
    if (answer.take()) return 1;
    publish_counters_kernel<<<1, 64, 0, s>>>(map->d.ctr, answer.words, answer.stamp);
    ASH_LAUNCH_CHECK();
    if (answer.wait(s, kHostCounters)) return 1;
    decode_counters(answer.words, c);
    lock.lock();
    if (asker == kOwnCall ||
        (map->changes == changes && (s == map->changed_on || map->replayed) && !map->counters_known)) {
        map->counters = c;
        counters_taken(map);
    }
    return 0;
}

// Inserts whose counters nobody read (deferred activations) between two looks
// at them for tombstone upkeep.
constexpr int kUpkeepEvery = 64;

int64_t rebuild_scratch_bytes(const ash_map* map) {
    const int64_t keys = (map->capacity * map->key_dim * 4 + 255) & ~int64_t{255};
    return keys + map->capacity * 8;
}

// keep at least a fifth of the slots truly empty -- of the bucket array, and
// of the second region on its own account (`general_used`: its entries and
// tombstones; it may be much smaller than the table)
bool should_rebuild(const ash_map* map, int64_t size, int64_t tombstones, int64_t incoming,
                    int64_t general_used = 0, int64_t general_tombstones = 0) {
    if (tombstones <= 0) return false;
    int64_t room = map->capacity - size;
    if (room < 0) room = 0;
    const int64_t arriving = incoming < room ? incoming : room;
    const int64_t slots = static_cast<int64_t>(map->d.nb) * kSlots;
    if ((size + tombstones + arriving) * 5 > slots * 4) return true;
    return map->general_attached && general_tombstones > 0 &&
           general_used * 5 > static_cast<int64_t>(map->d.gslots) * 4;
}

// Before an insert of `incoming` keys (the map's device is current, `s` is not
// being captured): if earlier erases or refused keys may have left
// tombstones, looks at the counters and re-places the live entries into an
// emptied table when too few empty slots would remain.
int upkeep(ash_map* map, int64_t incoming, void* scratch, int64_t scratch_bytes,
           hipStream_t s) {
    {
        std::lock_guard<std::mutex> lock(map->counter_lock);
        if (take_late_words(map)) return 1;
    }
    if (map->unread_inserts >= kUpkeepEvery || map->replayed) map->maybe_tombstones = true;
    if (!map->maybe_tombstones) return 0;
    ash_counters c;
    if (refresh_counters(map, s, kOwnCall, c)) return 1;
    map->maybe_tombstones = c.tombstones > 0;
    if (!should_rebuild(map, c.size, c.tombstones, incoming,
                        c.general_live + c.general_tombstones, c.general_tombstones)) {
        return 0;
    }
    int32_t* keys = nullptr;
    int64_t* indices = nullptr;
    // (after a load that has refused pairs the size is not the number of entries,
    // and what a listing leaves unwritten would be put back as well)
    if (map->general_attached && c.load_refused > 0) return 0;
    if (map->general_attached && c.size > 0) {
        // entries of the second region do not stand in the key log: the pairs
        // are listed into the caller's scratch and put back from there
        if (scratch == nullptr || scratch_bytes < rebuild_scratch_bytes(map)) {
            ASH_FAIL("scratch too small to re-place the entries: size it with "
                     "ash_map_insert_scratch_bytes before every insert");
        }
        keys = static_cast<int32_t*>(scratch);
        indices = reinterpret_cast<int64_t*>(
                static_cast<char*>(scratch) +
                ((map->capacity * map->key_dim * 4 + 255) & ~int64_t{255}));
    }
    if (ash_map_rebuild(map, keys, indices, c.size, s)) return 1;
    map->maybe_tombstones = false;
    c.tombstones = 0;
    std::lock_guard<std::mutex> lock(map->counter_lock);
    map->counters = c;
    map->counters_known = true;
    return 0;
}

}  // namespace

}  // extern "C"

int ash::queue_touched_count(ash_map* map, const uint8_t* touched, int64_t rows, int32_t* counts,
                             int max_counts, hipStream_t s) {
    LatePlace late(map);
    if (late.take(true)) return 1;
    int64_t groups = (rows + kCountFlags - 1) / kCountFlags;
    if (groups > max_counts) groups = max_counts;
    if (groups < 1) groups = 1;
    Change change(map, kChangeElse, s);
    count_flags_kernel<<<static_cast<unsigned>(groups), kCollectThreads, 0, s>>>(
            touched, rows, counts, map->d.ctr, late.late(), late.stamp);
    ASH_LAUNCH_CHECK();
    if (groups > 1) {
        publish_touched_kernel<<<1, kCollectThreads, 0, s>>>(
                map->d.ctr, counts, static_cast<int>(groups), late.late(), late.stamp);
        ASH_LAUNCH_CHECK();
    }
    change.queued();
    late.queued();
    return 0;
}

extern "C" {

int ash_map_set_staging(ash_map_t* map, int32_t* staging) {
    (void)staging;
    return check_map(map);
}

int ash_map_counters(ash_map_t* map, int32_t* staging, int64_t out[7], void* stream) {
    (void)staging;
    if (check_map(map)) return 1;
    if (out == nullptr) ASH_FAIL("null status output");
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    ash_counters c;
    if (refresh_counters(map, static_cast<hipStream_t>(stream), kReader, c)) return 1;
    out[0] = c.size;
    out[1] = c.dropped;
    out[2] = c.tombstones;
    out[3] = c.exotic_pending;
    out[4] = c.load_refused;
    out[5] = c.touched;
    out[6] = c.general_live;
    return 0;
}

int ash_map_counters_pending(ash_map_t* map) {
    if (map == nullptr) return 0;
    std::lock_guard<std::mutex> lock(map->counter_lock);
    return map->late_pending && !map->late_of_erase ? 1 : 0;
}

int ash_map_known_size(ash_map_t* map, int64_t* size) {
    if (check_map(map)) return -1;
    if (size == nullptr) {
        set_error("null size output");
        return -1;
    }
    if (map->replayed) return 0;
    std::lock_guard<std::mutex> lock(map->counter_lock);
    if (!map->counters_known) {
        if (!map->late_pending) return 0;
        DeviceGuard guard;
        if (guard.enter(map->device) != hipSuccess || take_late_words(map)) return -1;
    }
    *size = map->counters.size;
    return 1;
}

int ash_map_status(ash_map_t* map, int64_t out[5], void* stream) {
    if (check_map(map)) return 1;
    if (out == nullptr) ASH_FAIL("null status output");
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    // always a copy from the device
    ash_counters c;
    if (refresh_counters(map, static_cast<hipStream_t>(stream), kReaderOfDevice, c)) return 1;
    out[0] = c.size;
    out[1] = c.dropped;
    out[2] = c.tombstones;
    out[3] = c.exotic_pending;
    out[4] = c.load_refused;
    return 0;
}

int ash_map_upkeep(ash_map_t* map, int64_t incoming, void* scratch, int64_t scratch_bytes,
                   int32_t* staging, void* stream) {
    (void)staging;
    if (check_map(map)) return 1;
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (is_capturing(s)) return 0;
    return upkeep(map, incoming, scratch, scratch_bytes, s);
}

namespace {

// Which path an insert of this batch takes; *bytes = device scratch it needs.
enum { kPathPerKey = 0, kPathAssigned = 1, kPathStreaming = 2 };

int plan_insert(ash_map_t* map, int64_t n, int n_values, const int64_t* row_bytes, int policy,
                int* path, int64_t* bytes) {
    if (policy < ASH_STREAMING_AUTO || policy > ASH_STREAMING_EARLY) ASH_FAIL("unknown policy");
    if (n_values < 0) ASH_FAIL("negative value count");
    if (n_values > 0 && row_bytes == nullptr) ASH_FAIL("null value tables");
    *path = kPathPerKey;
    *bytes = 0;
    if (n_values > 0 && ash_map_insert_needs_scratch(n_values, row_bytes)) {
        *path = kPathAssigned;
        *bytes = n * 4;
    } else if (policy != ASH_STREAMING_NEVER) {
        int64_t ws = 0;
        int worthwhile = 0;
        if (ash_map_bulk_workspace_bytes(map, n, n_values, row_bytes, &ws, &worthwhile)) return 1;
        if (ws > 0 && (worthwhile || policy == ASH_STREAMING_ALWAYS ||
                       (policy == ASH_STREAMING_EARLY && streams_early(map, n, n_values)))) {
            *path = kPathStreaming;
            *bytes = ws;
        }
    }
    // a map with a second region re-places its entries through the scratch
    if (map->general_attached &&
        (map->maybe_tombstones || map->unread_inserts >= kUpkeepEvery || map->replayed)) {
        const int64_t r = rebuild_scratch_bytes(map);
        if (r > *bytes) *bytes = r;
    }
    return 0;
}

}  // namespace

int ash_map_insert_scratch_bytes(ash_map_t* map, int64_t n, int n_values,
                                 const int64_t* row_bytes, int policy, int64_t* bytes) {
    if (check_map(map)) return 1;
    if (bytes == nullptr) ASH_FAIL("null output pointer");
    if (n < 0) ASH_FAIL("negative key count");
    int path = 0;
    return plan_insert(map, n, n_values, row_bytes, policy, &path, bytes);
}

int ash_map_insert_auto(ash_map_t* map, const int32_t* keys, int64_t n, int n_values,
                        const void* const* src, void* const* dst, const int64_t* row_bytes,
                        void* scratch, int64_t scratch_bytes, int policy, int32_t* staging,
                        void* stream) {
    (void)staging;
    if (check_batch(map, keys, n)) return 1;
    if (n == 0) return 0;
    int path = 0;
    int64_t need = 0;
    if (plan_insert(map, n, n_values, row_bytes, policy, &path, &need)) return 1;
    if (need > 0 && (scratch == nullptr || scratch_bytes < need)) {
        ASH_FAIL("insert scratch too small: size it with ash_map_insert_scratch_bytes");
    }
    if (need > 0 && reinterpret_cast<uintptr_t>(scratch) % 256 != 0) {
        ASH_FAIL("insert scratch must be 256-byte aligned");
    }
    if (check_rows(n_values, src, dst, row_bytes)) return 1;
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool capturing = is_capturing(s);
    // (a capture replays launches only: no look at the counters, no upkeep;
    // refused keys stay in the counters for a later call to find)
    if (!capturing && upkeep(map, n, scratch, scratch_bytes, s)) return 1;
    if (path == kPathStreaming) {
        LatePlace late(map);
        if (!capturing && late.take(true)) return 1;
        // Only keys that the first pass hands to the per-key kernel can be
        // waiting for the second region; their number arrives a quarter into
        // the call's work.  None: the counters come with the insert's last
        // launch, and nobody waits for them here.
        bool published = false;
        if (insert_bulk(map, keys, n, n_values, src, dst, row_bytes, scratch, scratch_bytes,
                        capturing ? nullptr : late.early(), capturing ? nullptr : late.late(), late.stamp,
                        &published, stream)) {
            return 1;
        }
        if (capturing) return 0;
        if (published) {
            late.queued();
            return 0;
        }
        late.unused();
    } else {
        // The counters come behind the insert (a short launch leaves them itself) and
        // wait for the call that asks for them; only a batch with keys for the second
        // region, which may be missing or full, is waited for here.  (Under the other
        // policies callers find the counters read.  Replays change them behind the
        // host's back: read, too.)
        if (capturing || map->replayed || policy != ASH_STREAMING_EARLY) {
            // (short launches leave what is waited for below themselves)
            Answer answer;
            Publish publish = {};
            if (!capturing && n <= kLeaveKeys) {
                if (answer.take()) return 1;
                publish = {answer.words, answer.stamp, next_ticket(map)};
            }
            if (insert_per_key(map, keys, n, n_values, src, dst, row_bytes,
                               path == kPathAssigned ? static_cast<int32_t*>(scratch) : nullptr,
                               stream, publish)) {
                answer.abandon();   // (the launch may have been made)
                return 1;
            }
            if (capturing) return 0;
            if (publish.landing != nullptr) {
                if (answer.wait(s, kHostCounters)) return 1;
                std::lock_guard<std::mutex> lock(map->counter_lock);
                decode_counters(answer.words, map->counters);
                counters_taken(map);
            }
        } else {
            Answer answer;
            KeyCheck check = {};
            if (map->key_dim > 1) {
                if (answer.take()) return 1;
                const int64_t groups = (n + kCheckKeys * kHeapBlock - 1) / (kCheckKeys * kHeapBlock);
                check = {static_cast<unsigned>(std::min<int64_t>(groups, kMostChecks)), answer.words,
                         answer.stamp, next_ticket(map)};
            }
            LatePlace late(map);
            if (late.take(true)) return 1;
            // (the words of the answer may come from any exit below that follows a launch)
            if (check.groups > 0) answer.abandon();
            const bool leaves = n <= kLeaveKeys;
            Publish publish = {};
            if (leaves) publish = {late.late(), late.stamp, next_ticket(map)};
            if (insert_per_key(map, keys, n, n_values, src, dst, row_bytes,
                               path == kPathAssigned ? static_cast<int32_t*>(scratch) : nullptr,
                               stream, publish, check)) {
                return 1;
            }
            if (!leaves) {
                publish_counters_kernel<<<1, 64, 0, s>>>(map->d.ctr, late.late(), late.stamp);
                ASH_LAUNCH_CHECK();
            }
            late.queued();
            if (check.groups == 0) return 0;
            if (answer.wait(s, 1)) return 1;
            if (value_of(answer.words[0]) == 0) return 0;
        }
    }
    ash_counters c;
    if (refresh_counters(map, s, kOwnCall, c)) return 1;
    if (c.exotic_pending > 0 && map->general_attached) {
        Change change(map, kChangeElse, s);
        fold_waiting_keys_kernel<<<1, 64, 0, s>>>(map->d.ctr);
        ASH_LAUNCH_CHECK();
        c.dropped += c.exotic_pending;
        c.exotic_pending = 0;
        change.queued_with(c);
        map->maybe_tombstones = true;
    }
    if (c.exotic_pending > 0) {
        set_error("keys that do not fit the packed code are waiting for the second region: "
                  "attach it (ash_map_attach_general) and issue the insert again");
        return ASH_NEEDS_GENERAL;
    }
    return 0;
}

int ash_map_erase_scratch_bytes(ash_map_t* map, int64_t n, int policy, int64_t* bytes) {
    if (check_map(map)) return 1;
    if (bytes == nullptr) ASH_FAIL("null output pointer");
    if (policy < ASH_STREAMING_AUTO || policy > ASH_STREAMING_NEVER) ASH_FAIL("unknown policy");
    *bytes = 0;
    if (policy == ASH_STREAMING_NEVER) return 0;
    int64_t ws = 0;
    int worthwhile = 0;
    if (ash_map_erase_bulk_query(map, n, &ws, &worthwhile)) return 1;
    if (ws > 0 && (worthwhile || policy == ASH_STREAMING_ALWAYS)) *bytes = ws;
    return 0;
}

int ash_map_erase_auto(ash_map_t* map, const int32_t* keys, int64_t n, void* scratch,
                       int64_t scratch_bytes, int policy, void* stream) {
    if (check_batch(map, keys, n)) return 1;
    if (n == 0) return 0;
    int64_t need = 0;
    if (ash_map_erase_scratch_bytes(map, n, policy, &need)) return 1;
    if (need == 0) return ash_map_erase(map, keys, n, stream);
    if (scratch == nullptr || scratch_bytes < need) {
        ASH_FAIL("erase scratch too small: size it with ash_map_erase_scratch_bytes");
    }
    return ash_map_erase_bulk(map, keys, n, scratch, scratch_bytes, stream);
}

int ash_grid_collect_touched(ash_map_t* map, uint8_t* touched, const int32_t* block_coords,
                             int64_t* out_indices, int32_t* out_coords, void* stream) {
    if (check_map(map)) return 1;
    if (touched == nullptr || block_coords == nullptr || out_indices == nullptr ||
        out_coords == nullptr) {
        ASH_FAIL("null pointer in grid_collect_touched");
    }
    if (map->capacity > kCollectMaxBlocks) ASH_FAIL("grid_collect_touched: more than ASH_COLLECT_MAX_BLOCKS rows");
    if (reinterpret_cast<uintptr_t>(touched) % 4 != 0) ASH_FAIL("grid_collect_touched: flags must be 4-byte aligned");
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    const int64_t per_group = int64_t{4} * kCollectThreads;   // flags of a one-word-per-thread chunk
    int64_t groups = (map->capacity + per_group - 1) / per_group;
    if (groups > kCollectGroups) groups = kCollectGroups;
    const int words = static_cast<int>((map->capacity + groups * per_group - 1) / (groups * per_group));
    groups = (map->capacity + words * per_group - 1) / (words * per_group);   // no empty chunks
    Change change(map, kChangeElse, static_cast<hipStream_t>(stream));   // the number of listed rows is a counter
    collect_touched_kernel<<<static_cast<unsigned>(groups), kCollectThreads, 0,
                             static_cast<hipStream_t>(stream)>>>(
            touched, block_coords, map->capacity, words, out_indices, out_coords, map->d.ctr);
    ASH_LAUNCH_CHECK();
    return 0;
}

int ash_map_size(ash_map_t* map, int64_t* size, void* stream) {
    if (size == nullptr) ASH_FAIL("null size output");
    int64_t c[7];
    if (ash_map_counters(map, nullptr, c, stream)) return 1;
    *size = c[0];
    return 0;
}

int ash_map_items(ash_map_t* map, int32_t* keys_out, int64_t* indices_out,
                  int64_t n_expected, void* stream) {
    return ash_map_items_rows(map, keys_out, indices_out, n_expected, 0, nullptr, nullptr, nullptr,
                              nullptr, stream);
}

int ash_map_items_rows(ash_map_t* map, int32_t* keys_out, int64_t* indices_out, int64_t n_expected,
                       int n_values, const void* const* src, void* const* dst,
                       const int64_t* row_bytes, const int64_t* src_rows, void* stream) {
    if (check_map(map)) return 1;
    if (n_expected < 0) ASH_FAIL("negative item count");
    if (n_values < 0 || n_values > kMaxFusedValues) ASH_FAIL("items: up to 4 value tables per call");
    if (n_expected == 0) return 0;
    if (keys_out == nullptr || indices_out == nullptr) {
        ASH_FAIL("null output pointer");
    }
    GatherArgs rows = {};
    int64_t most = 0;
    if (n_values > 0 && gather_args(n_values, src, dst, row_bytes, src_rows, n_expected, rows, most)) return 1;
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (settle_table(map, s)) return 1;
    const int identity = heap_in_order(map) ? 1 : 0;
    const bool all_in_log = none_in_general(map);
    if (identity && all_in_log) {
        const int64_t n = n_expected < map->capacity ? n_expected : map->capacity;
        const unsigned gd = grid_for(n);
        switch (map->key_dim) {
            case 1:
                items_dense_kernel<1><<<gd, kBlock, 0, s>>>(map->d, keys_out, indices_out, n);
                break;
            case 2:
                items_dense_kernel<2><<<gd, kBlock, 0, s>>>(map->d, keys_out, indices_out, n);
                break;
            case 3:
                items_dense_kernel<3><<<gd, kBlock, 0, s>>>(map->d, keys_out, indices_out, n);
                break;
            default:
                items_dense_kernel<4><<<gd, kBlock, 0, s>>>(map->d, keys_out, indices_out, n);
                break;
        }
        ASH_LAUNCH_CHECK();
        return n_values > 0 ? ash_gather_rows(n_values, src, dst, row_bytes, src_rows, nullptr, n, stream) : 0;
    }
    // Rows go along with the entries that the log lists, up to the width at which a
    // lane copies one word after the other; entries of the second region are not
    // listed there.
    bool along = all_in_log;
    for (int v = 0; v < n_values; ++v) along = along && rows.row_dwords[v] <= kMaxFusedRowDwords;
    if (!along) rows.n = 0;
    const int slot = next_slot(map);
    switch (map->key_dim) {
        case 1:
            launch_items<1>(map, keys_out, indices_out, n_expected, identity, rows, slot, all_in_log, s);
            break;
        case 2:
            launch_items<2>(map, keys_out, indices_out, n_expected, identity, rows, slot, all_in_log, s);
            break;
        case 3:
            launch_items<3>(map, keys_out, indices_out, n_expected, identity, rows, slot, all_in_log, s);
            break;
        default:
            launch_items<4>(map, keys_out, indices_out, n_expected, identity, rows, slot, all_in_log, s);
            break;
    }
    ASH_LAUNCH_CHECK();
    if (!all_in_log) {
        const unsigned gg = grid_for(map->d.gslots);
        int32_t* cursor = map->d.ctr + kCtrCursors + 2 * slot;   // its lower half
        auto kernel = map->key_dim == 1   ? items_general_kernel<1>
                      : map->key_dim == 2 ? items_general_kernel<2>
                      : map->key_dim == 3 ? items_general_kernel<3>
                                          : items_general_kernel<4>;
        kernel<<<gg, kBlock, 0, s>>>(map->d, keys_out, indices_out, n_expected, cursor);
        ASH_LAUNCH_CHECK();
        for (int half = 0; half < 2; ++half) {
            set_counter_kernel<<<1, 64, 0, s>>>(cursor, half, 0);
            ASH_LAUNCH_CHECK();
        }
    }
    if (n_values > 0 && !along) {
        return ash_gather_rows(n_values, src, dst, row_bytes, src_rows, indices_out, n_expected, stream);
    }
    return 0;
}

int ash_map_should_rebuild(ash_map_t* map, int64_t size, int64_t tombstones,
                           int64_t incoming) {
    if (map == nullptr) return 0;
    return should_rebuild(map, size, tombstones, incoming) ? 1 : 0;
}

int ash_map_rebuild(ash_map_t* map, int32_t* keys_scratch,
                    int64_t* indices_scratch, int64_t n, void* stream) {
    if (check_map(map)) return 1;
    if (n < 0 || n > map->capacity) ASH_FAIL("rebuild: bad entry count");
    // Without a second region every entry stands in the key log under its
    // index and is put back from there; with one, the pairs are listed into the
    // caller's scratch first.
    const bool from_log = !map->general_attached;
    if (!from_log && n > 0 && (keys_scratch == nullptr || indices_scratch == nullptr)) {
        ASH_FAIL("rebuild: null scratch pointer");
    }
    if (!from_log && n > 0 && ash_map_items(map, keys_scratch, indices_scratch, n, stream)) {
        return 1;
    }
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    Change change(map, kChangeElse, s);
    if (fill_buckets(map, s)) return 1;
    if (map->general_attached) {
        const int64_t g16 = static_cast<int64_t>(map->d.gslots) / 4;
        fill16_kernel<<<capped_grid(g16), kBlock, 0, s>>>(
                reinterpret_cast<uint4*>(map->d.gstate), g16, 0xFFFFFFFFu);
        ASH_LAUNCH_CHECK();
        set_counter_kernel<<<1, 64, 0, s>>>(map->d.ctr, kCtrGenLive, 0);   // counted again below
        ASH_LAUNCH_CHECK();
        set_counter_kernel<<<1, 64, 0, s>>>(map->d.ctr, kCtrGenTombs, 0);
        ASH_LAUNCH_CHECK();
    }
    set_counter_kernel<<<1, 64, 0, s>>>(map->d.ctr, kCtrTombs, 0);
    ASH_LAUNCH_CHECK();
    if (n == 0) return 0;
    if (from_log) {
        int64_t g = (map->capacity + kHeapBlock - 1) / kHeapBlock;
        if (g > 256 * 16) g = 256 * 16;
        replace_from_log_kernel<<<static_cast<unsigned>(g), kHeapBlock, 0, s>>>(
                map->d, heap_in_order(map) ? 1 : 0);
        ASH_LAUNCH_CHECK();
        return 0;
    }
    ValueArgs va = {};
    return launch_insert_to<kInsertLoad, false>(map, keys_scratch, n, va, nullptr,
                                                indices_scratch, s);
}

int ash_map_neighbors(ash_map_t* map, int64_t num_rows, int radius, int bidirectional,
                      int32_t* coords, int64_t* lut, void* stream) {
    if (check_map(map)) return 1;
    if (map->key_dim != 3) ASH_FAIL("neighbour tables need three-dimensional keys");
    if (num_rows < 0 || radius < 0 || radius > 15) ASH_FAIL("neighbour table: bad sizes");
    if (num_rows == 0) return 0;
    if (coords == nullptr || lut == nullptr) ASH_FAIL("null output pointer");
    const NeighborArgs a = {coords, lut, num_rows, bidirectional ? 2 * radius + 1 : radius + 1,
                            bidirectional ? radius : 0};
    const int64_t each = static_cast<int64_t>(a.width) * a.width * a.width;
    if (num_rows > (int64_t{1} << 39) / each - kBlock) ASH_FAIL("neighbour table: too many rows");
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (settle_table(map, s)) return 1;
    const auto kernel = a.width == 2 ? neighbors_kernel<2> : a.width == 3 ? neighbors_kernel<3> : neighbors_kernel<0>;
    kernel<<<grid_for(num_rows * each), kBlock, 0, s>>>(map->d, a, heap_in_order(map) ? 1 : 0);
    ASH_LAUNCH_CHECK();
    if (!none_in_general(map)) {
        neighbors_general_kernel<<<looping_grid(map->d.gslots * each), kBlock, 0, s>>>(map->d, a);
        ASH_LAUNCH_CHECK();
    }
    return 0;
}

int ash_map_items_in_index_order(ash_map_t* map, int* dense) {
    if (check_map(map)) return 1;
    if (dense == nullptr) ASH_FAIL("null output pointer");
    *dense = lists_in_index_order(map) ? 1 : 0;
    return 0;
}

int ash_map_load(ash_map_t* map, const int32_t* keys, const int64_t* indices,
                 int64_t n, const int32_t* heap_src, void* stream) {
    if (check_batch(map, keys, n)) return 1;
    if (n > map->capacity) ASH_FAIL("more pairs than capacity");
    if (n > 0 && indices == nullptr) ASH_FAIL("null indices pointer");
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (is_capturing(s)) ASH_FAIL("ash_map_load cannot be captured into a graph");
    Change change(map, kChangeElse, s);
    if (clear_table(map, s, false, static_cast<int32_t>(n))) return 1;
    map->heap_dirty = true;   // the heap is the caller's from here on
    map->maybe_tombstones = false;
    map->unread_inserts = 0;
    if (heap_src != nullptr && heap_src != map->d.heap) {
        ASH_HIP(hipMemcpyAsync(map->d.heap, heap_src,
                               static_cast<size_t>(map->capacity) * 4,
                               hipMemcpyDeviceToDevice, s));
    }
    // later inserts take their indices from this heap unchecked
    check_heap_kernel<<<looping_grid(map->capacity), kBlock, 0, s>>>(map->d.heap, map->capacity,
                                                                   map->d.ctr);
    ASH_LAUNCH_CHECK();
    if (n == 0) return 0;
    ValueArgs va = {};
    return launch_insert_to<kInsertLoad, false>(map, keys, n, va, nullptr, indices, s);
}

}  // extern "C"
