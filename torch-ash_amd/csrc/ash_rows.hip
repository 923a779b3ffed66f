// Backward and backward of the backward of the trilinear query by rows: the kernels
// that give a lane a whole query (rows_by_lane in ash_query.hip says which go this way).
//
// Compiled once for every width, -DASH_ROW_WIDTH=<channels>, each into device code of
// its own: the runtime loads that of a source file when the first of its kernels is
// launched, and a program that trains rows of one width has 0.4 of 4 MB to wait for, one
// that only interpolates none (all widths beside the forward kernels -> so: first
// interpolation of a process 25 -> 11.8 ms, the training pass after it 7.1 -> 8.7).
#include "ash_query.h"

#ifndef ASH_ROW_WIDTH
#error "ASH_ROW_WIDTH: the number of channels to compile for"
#endif

namespace ash {
namespace {

// Wavefronts per SIMD that the kernels are compiled for.  Two workgroups of eight, which
// the line tables leave room for, want 128 registers at most: both gradients of seven and
// eight channels, which take 123 - 139 else (rows of seven 151 -> 118 us, for 8 bytes of
// scratch a lane; eight, 32 and 60; up to six take fewer anyway).  Twelve, held to 168 by
// three, spill 8 and, both orders with the positions' gradient, 60 bytes.
constexpr int kWavesRows = 3;
constexpr int waves_of_rows(int E, int threads) { return threads > 256 && (E == 7 || E == 8) ? 4 : kWavesRows; }

// Workgroups of four wavefronts that are on a CU at once by their registers (the fifth of
// 96, the fourth of 128, the third of 168; LDS leaves room for four with line tables): a
// persistent grid of more is not all under way from the start.  `order` 1: the backward,
// 2: that of the backward; `out`: what is asked for, as the kernels have it.  With four
// where three fit: 500 000 ray samples, both orders with the positions' gradient and second
// order with grad_z, of seven channels 82 -> 68 and 76 -> 64 us, of eight 70 -> 58 and 68 ->
// 57; grad_z alone with six where five fit and four where three: 1.3 M of six 77 -> 70,
// 660 000 of twelve 56 -> 53.
constexpr int resident_rows(int E, int order, int out) {
    if ((out & 1) != 0) return (out & 2) == 0 || E < 7 || (E <= 8 && order == 1 && out == 3) ? 4 : 3;
    if (order == 1) return E <= 5 ? 8 : E == 6 ? 7 : E == 7 ? 5 : E <= 12 ? 4 : 3;
    return E <= 3 ? 8 : E == 4 ? 7 : E == 5 ? 6 : E <= 7 ? 5 : E == 8 ? 4 : 3;
}

// ================================================= backward kernels by rows
// fp32 rows of few channels (rows_by_lane): one lane holds a whole query, as in the
// forward kernel, so that a wavefront serves 64 queries per tile: four channels have four
// times the loads in flight and a quarter of the per-query arithmetic of the
// one-lane-per-channel kernels of ash_query.hip, and rows of five leave no lanes idle.
//
// Gradient rows.  The memory side executes atomics at a fixed rate of
// requests, and one request is what one instruction of a wavefront sends to
// one 64-byte line, whether it carries one float or sixteen (measured: 18 G
// requests/s for 4-byte and for 64-byte groups alike).  The eight corners of a
// query and the queries that follow it along a ray meet the same few lines
// over and over -- the x neighbour is the next row, a corner of this sample is
// another corner of the next -- but in different instructions.  So every
// wavefront first adds its contributions into a small table of lines in LDS
// (open addressing on the line number, sixteen floats per entry; a row may end in the
// line after the one it starts in) and sends the
// table out once per tile, one line per sixteen lanes: a third of the requests
// on ray-ordered samples.  Before that, runs of consecutive queries with the
// same row are summed in registers (lane exchange inside a row of 16 lanes is
// a modifier of an ordinary vector instruction, across rows it would be a trip
// through the LDS pipeline, so a run is cut at the row of lanes; the table
// joins the pieces).  A row whose line finds no place within kLineProbes steps
// goes to memory directly, and a wavefront that sent more rows that way than
// the table has lines leaves the table aside for the next kLineRest tiles.
//
// Queries in no order share no lines but those of neighbouring corners.  A tile of which
// more than half lie in another block than the query before them leaves the table aside
// at once: the rows of two corners that differ in x follow each other in memory, and leave
// together by neighbouring lanes of one instruction, five requests for eight rows of four
// channels (rows of one by one through the table until it had rested: 398 -> 273 us for
// 1 M unordered queries of four channels, 17 -> 7 for 1000).  Ordered tiles do not pay for
// it: second order and both orders of four channels, without the test and the rows past
// the table -> with them, 131 000 12.5 -> 12.3, 400 000 34.9 -> 34.8, 4 M 248 -> 248.
// Every corner with a copy of its code: one copy for all, which selects its row and its
// terms, takes half as long again (131 000 of four channels 13 -> 19 us), and a second pass
// for the rows past the table 14.6.
template <int CTRL>
__device__ __forceinline__ int dpp_int(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}
template <int CTRL, typename T>
__device__ __forceinline__ T dpp(T v) {
    static_assert(sizeof(T) == 4, "32-bit values");
    return __builtin_bit_cast(T, dpp_int<CTRL>(__builtin_bit_cast(int, v)));
}
constexpr int kRowShl = 0x100;  // lane i takes lane i + n of its row of 16 (0 beyond it)
constexpr int kRowShr = 0x110;  // lane i takes lane i - n

constexpr int kRowBcast15 = 0x142;  // every lane of a row takes lane 15 of the row before

// Runs of consecutive lanes whose queries lie in the same cell.  Two queries
// meet in the same row at a corner only when they lie in the same cell, and
// then at every corner, so the runs are found once per tile, from the row of the
// cell itself, and the sums over them are taken corner by corner (sum_runs).
// The sums run inside the rows of 16 lanes; a run that goes on in the next row
// hands its part over: lane 15 keeps quiet and the lane that ends the run in
// the next row adds what lane 15 had.  (A run that fills a whole row and still
// goes on is not handed over a second time; its parts meet in the table of
// lines.)
struct Runs {
    bool any;         // some lane continues the run of the lane before it (the same for all lanes)
    bool take[4];     // step 1, 2, 4, 8 of the segmented sum adds what lies that far below
    bool takes_offer; // adds what lane 15 of the row before holds
    bool tail;        // this lane ends its run and holds the total
    bool ordered;     // half of the queries are less than a block's cells from the one before (the same for all lanes)
};

// The runs of a tile.  Lanes without a query (not `on`) get a number no neighbour shares.
// `cells`: of a block.  Every lane of the wavefront must take part.
__device__ __forceinline__ Runs find_runs(uint32_t cell_row, bool on, uint32_t cells, int lane) {
    Runs r;
    const uint32_t id = on ? cell_row : (kNoRow - static_cast<uint32_t>(lane & 1));
    const int g = lane & 15;
    const uint32_t prev = dpp<kRowShr + 1>(id);
    const uint32_t ahead = id - prev, behind = prev - id;
    const uint64_t queries = __builtin_amdgcn_ballot_w64(on);
    const uint64_t near = __builtin_amdgcn_ballot_w64((ahead < behind ? ahead : behind) < cells);
    r.ordered = 2 * __popcll(near & queries) >= __popcll(queries);
    const uint32_t next = dpp<kRowShl + 1>(id);
    const bool joins = g > 0 && prev == id;
    r.any = __ballot(joins) != 0;
    const bool starts = g > 0 && prev != id;   // a run starts here, inside the row
    int f = (g == 0 || starts) ? 1 : 0;        // a run starts at or below this lane, as far as summed
    {
        const int fu = dpp_int<kRowShr + 1>(f);
        r.take[0] = g >= 1 && !f;
        if (r.take[0]) f |= fu;
    }
    {
        const int fu = dpp_int<kRowShr + 2>(f);
        r.take[1] = g >= 2 && !f;
        if (r.take[1]) f |= fu;
    }
    {
        const int fu = dpp_int<kRowShr + 4>(f);
        r.take[2] = g >= 4 && !f;
        if (r.take[2]) f |= fu;
    }
    r.take[3] = g >= 8 && !f;
    bool tail = g == 15 || next != id;
    // in the first run of its row: no run starts between the row's first lane and here
    const uint64_t started = __ballot(starts);
    const uint64_t upto = (2ull << lane) - 1ull;
    const uint64_t row_lanes = 0xFFFFull << (lane & 48);
    const bool first_run = (started & upto & row_lanes) == 0;
    // lane 15 offers its sum unless its run began with the row
    const int offers = (g == 15 && !first_run) ? 1 : 0;
    const int offered = dpp_int<kRowBcast15>(offers);
    const uint32_t offered_id = dpp<kRowBcast15>(id);
    r.takes_offer = lane >= 16 && tail && first_run && offered != 0 && offered_id == id;
    // ... and keeps quiet when the next row takes the offer
    const uint32_t id16 = __builtin_amdgcn_readlane(id, 16);
    const uint32_t id32 = __builtin_amdgcn_readlane(id, 32);
    const uint32_t id48 = __builtin_amdgcn_readlane(id, 48);
    const uint32_t over = lane < 16 ? id16 : lane < 32 ? id32 : id48;
    if (offers != 0 && lane < 48 && over == id) tail = false;
    r.tail = tail;
    return r;
}

template <int D, int E>
__device__ __forceinline__ void run_step(float (&v)[E], bool take) {
#pragma unroll
    for (int k = 0; k < E; ++k) {
        const float vu = dpp<kRowShr + D>(v[k]);
        if (take) v[k] += vu;
    }
}

// Sums `v` over the runs; the lanes with r.tail hold the totals afterwards.
// Every lane of the wavefront must take part.
template <int E>
__device__ __forceinline__ void sum_runs(const Runs& r, float (&v)[E]) {
    run_step<1>(v, r.take[0]);
    run_step<2>(v, r.take[1]);
    run_step<4>(v, r.take[2]);
    run_step<8>(v, r.take[3]);
#pragma unroll
    for (int k = 0; k < E; ++k) {
        const float part = dpp<kRowBcast15>(v[k]);
        if (r.takes_offer) v[k] += part;
    }
}

constexpr int kLineSlots = 128;   // lines per wavefront's table
constexpr int kLineProbes = 4;
constexpr int kLineRest = 7;
// Lanes that a row leaves past the table by, and rows of one instruction (of one
// channel: of a quarter of its lanes, for which there is room)
constexpr int line_out_lanes(int E) { return E <= 4 ? 4 : E <= 8 ? 8 : 16; }
constexpr int line_out_rows(int E) { return 64 / line_out_lanes(E); }
constexpr uint32_t kLineFree = 0xFFFFFFFFu;
// float k of slot h sits at k * kLinePitch + h: the sixteen floats of a line
// and the same float of neighbouring slots fall into different banks
constexpr int kLinePitch = kLineSlots + 1;

struct LineTable {
    float val[16 * kLinePitch];
    uint32_t key[kLineSlots];
    // rows on their way to memory without the table; the flush keeps its list
    // of used slots in the same place
    union {
        struct {
            uint32_t row[16];
            float v[64];
        } out;
        uint8_t used[kLineSlots];
    };
};

// Orders the LDS traffic of one wavefront (whose LDS instructions execute in
// program order, each for all its lanes) for the compiler.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The floats of a row added to their places in LDS, `at(k)` for the k-th.  The LDS
// executes a floating-point add atomic one lane after the other (about three cycles a
// lane, measured) and a 32-bit compare-and-swap at full rate: the add is a read
// and a compare-and-swap of the sum.  The floats go side by side, two
// round trips for all of them; lanes that met another lane's update in between
// (seldom: runs of equal rows have been summed before) repeat float by float.
template <int E, typename At>
__device__ __forceinline__ void lds_add(At at, const float (&v)[E]) {
    unsigned int seen[E], got[E];
#pragma unroll
    for (int k = 0; k < E; ++k) seen[k] = *at(k);
#pragma unroll
    for (int k = 0; k < E; ++k) {
        got[k] = atomicCAS(at(k), seen[k], __float_as_uint(__uint_as_float(seen[k]) + v[k]));
    }
    bool done = true;
#pragma unroll
    for (int k = 0; k < E; ++k) done = done && got[k] == seen[k];
    if (done) return;
#pragma unroll 1
    for (int k = 0; k < E; ++k) {
        // (selects, not an indexed access: the arrays stay in registers)
        unsigned int g = got[0], s = seen[0];
        float add = v[0];
#pragma unroll
        for (int q = 1; q < E; ++q) {
            g = k == q ? got[q] : g;
            s = k == q ? seen[q] : s;
            add = k == q ? v[q] : add;
        }
        while (g != s) {
            s = g;
            g = atomicCAS(at(k), s, __float_as_uint(__uint_as_float(s) + add));
        }
    }
}

// Line of a row's first float, and where in it that stands.
template <int E>
__device__ __forceinline__ void line_of(uint32_t row, uint32_t& line, uint32_t& pos) {
    if constexpr (16 % E == 0) {
        line = row / (16 / E);
        pos = row % (16 / E) * E;
    } else {
        const uint64_t first = static_cast<uint64_t>(row) * E;
        line = static_cast<uint32_t>(first >> 4);
        pos = static_cast<uint32_t>(first) & 15u;
    }
}

struct LineAcc {
    LineTable* tab;
    int rest;      // tiles left during which the table is left aside
    int spilled;   // rows that found no place in the table since the last flush (whole wavefront)
    bool aside;    // the table is left aside during this tile, and its place used otherwise
    bool ready;    // the table is empty and its floats are zero (at the start of a tile)

    __device__ __forceinline__ void start(LineTable* t, int lane) {
        tab = t;
        rest = 0;
        spilled = 0;
        if (tab != nullptr) empty(lane);
    }

    __device__ __forceinline__ void empty(int lane) {
        for (int i = lane; i < 16 * kLinePitch; i += 64) tab->val[i] = 0.f;
        tab->key[lane] = kLineFree;
        tab->key[lane + 64] = kLineFree;
        wave_lds_fence();
        ready = true;
    }

    // Whole wavefront, before the first row of a tile.
    __device__ __forceinline__ void tile(bool ordered, int lane) {
        aside = rest > 0 || !ordered;
        if (!aside && !ready) empty(lane);
    }

    // Whether `line` finds a place, and its slot.  (Told by a flag: where the loop returns
    // the slot, it is four blocks with two branches a probe instead of one, in the chain that
    // a launch waits for: second order of 131 000 of four channels 13.2 us, so 12.3, of five
    // 17.8 -> 16.3; both orders of 400 000 of four 36.1 -> 34.8, of 1.6 M of five 140 -> 137.)
    __device__ __forceinline__ bool slot_of(uint32_t line, uint32_t& h) {
        bool placed = false;
        h = (line * 0x9E3779B1u) >> 25;
#pragma unroll 1
        for (int p = 0; p < kLineProbes; ++p) {
            const uint32_t old = atomicCAS(&tab->key[h], kLineFree, line);
            if (old == kLineFree || old == line) {
                placed = true;
                break;
            }
            h = (h + 1) & (kLineSlots - 1);
        }
        return placed;
    }

    // grad[E * row .. E * row + E - 1] += v for the lanes that `want`; every lane
    // of the wavefront must take part.
    template <int E>
    __device__ __forceinline__ void add(float* __restrict__ grad, bool want, uint32_t row,
                                        const float (&v)[E], int lane) {
        bool placed = false;
        if (want) {
            uint32_t line, pos;
            line_of<E>(row, line, pos);
            uint32_t h;
            placed = slot_of(line, h);
            if constexpr (16 % E == 0) {
                unsigned int* at = reinterpret_cast<unsigned int*>(tab->val + pos * kLinePitch + h);
                if (placed) lds_add<E>([&](int k) { return at + k * kLinePitch; }, v);
            } else {
                // a row may end in the next line (a line that was claimed for it alone
                // and stays empty where this one finds no place sends nothing)
                uint32_t next = h;
                if (placed && pos + E > 16u) placed = slot_of(line + 1u, next);
                unsigned int* at = reinterpret_cast<unsigned int*>(tab->val + pos * kLinePitch + h);
                const int over = static_cast<int>(next) - static_cast<int>(h) - 16 * kLinePitch;
                if (placed) {
                    lds_add<E>([&](int k) { return at + k * kLinePitch + (pos + k > 15u ? over : 0); }, v);
                }
            }
        }
        // The rest goes to memory now, regrouped so that the floats of a
        // row leave from neighbouring lanes of one instruction (one request a
        // row; one lane sending its floats would make as many).
        const uint64_t out = __ballot(want && !placed);
        if (out == 0) return;
        constexpr int kLanes = line_out_lanes(E), kRows = line_out_rows(E);
        const int n = __popcll(out);
        const int mine = __popcll(out & ((1ull << lane) - 1ull));
        spilled += n;
        for (int i = 0; i < n; i += kRows) {
            const int at = mine - i;
            wave_lds_fence();
            if (want && !placed && at >= 0 && at < kRows) {
                tab->out.row[at] = row;
                if constexpr (E == 4) {
                    *reinterpret_cast<float4*>(tab->out.v + at * 4) = make_float4(v[0], v[1], v[2], v[3]);
                } else {
#pragma unroll
                    for (int k = 0; k < E; ++k) tab->out.v[at * kLanes + k] = v[k];
                }
            }
            wave_lds_fence();
            const int e = lane / kLanes, k = lane % kLanes;
            if (i + e < n && k < E) {
                unsafeAtomicAdd(grad + static_cast<uint64_t>(tab->out.row[e]) * E + k, tab->out.v[lane]);
            }
        }
        wave_lds_fence();
    }

    // The same past the table, which is left aside and leaves room for all rows of two
    // corners: these follow each other in memory as a rule, and leave together.
    template <int E>
    __device__ __forceinline__ void send_two(float* __restrict__ grad, bool want, const uint32_t (&row)[2],
                                             const float (&v)[2][E], int lane) {
        constexpr int kPitch = 2 * E + 1, kAtOnce = 64 / (2 * E);
        static_assert(64 * (kPitch + 2) <= 16 * kLinePitch, "128 rows and their numbers");
        const uint64_t out = __ballot(want);
        const int n = __popcll(out);
        const int mine = __popcll(out & ((1ull << lane) - 1ull));
        uint32_t* const rows = reinterpret_cast<uint32_t*>(tab->val);
        float* const floats = tab->val + 128;
        wave_lds_fence();
        if (want) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                rows[2 * mine + h] = row[h];
#pragma unroll
                for (int k = 0; k < E; ++k) floats[mine * kPitch + h * E + k] = v[h][k];
            }
        }
        wave_lds_fence();
        const int e = lane / (2 * E), at = lane % (2 * E);
        const int half = at >= E ? 1 : 0, k = at - half * E;
        for (int i = e; i < n && e < kAtOnce; i += kAtOnce) {
            unsafeAtomicAdd(grad + static_cast<uint64_t>(rows[2 * i + half]) * E + k, floats[i * kPitch + at]);
        }
    }

    // Whole wavefront: sends the table's lines out and empties it.
    __device__ __forceinline__ void flush(float* __restrict__ grad, int lane) {
        wave_lds_fence();
        const bool lo = tab->key[lane] != kLineFree;
        const bool hi = tab->key[lane + 64] != kLineFree;
        const uint64_t mlo = __ballot(lo), mhi = __ballot(hi);
        const uint64_t below = (1ull << lane) - 1ull;
        const int nlo = __popcll(mlo);
        const int n = nlo + __popcll(mhi);
        if (lo) tab->used[__popcll(mlo & below)] = static_cast<uint8_t>(lane);
        if (hi) tab->used[nlo + __popcll(mhi & below)] = static_cast<uint8_t>(lane + 64);
        wave_lds_fence();
        // four lines per instruction, sixteen lines per turn: the reads of
        // a turn are issued together
        for (int i = 0; i < n; i += 16) {
            uint32_t h[4], line[4];
            float v[4];
            float* at[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = i + j * 4 + (lane >> 4);
                h[j] = e < n ? tab->used[e] : 0u;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = i + j * 4 + (lane >> 4);
                at[j] = tab->val + (lane & 15) * kLinePitch + h[j];
                line[j] = tab->key[h[j]];
                v[j] = e < n ? *at[j] : 0.f;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                // floats nobody contributed to are zero
                if (v[j] != 0.f) {
                    *at[j] = 0.f;
                    unsafeAtomicAdd(
                            grad + ((static_cast<uint64_t>(line[j]) << 4) | (lane & 15)), v[j]);
                }
            }
        }
        wave_lds_fence();
        tab->key[lane] = kLineFree;
        tab->key[lane + 64] = kLineFree;
        wave_lds_fence();
    }

    // The tile is done with.
    __device__ __forceinline__ void done() {
        if (aside) ready = false;
        if (rest > 0) {
            --rest;
        } else if (spilled > kLineSlots) {
            rest = kLineRest;   // more rows went past the table than it has lines
        }
        spilled = 0;
    }
};

// Waits here for what a load brings, in front of the two ways that scatter_rows goes: where
// either waited by itself, the first loads of the next tile waited for it once more, one by
// one, and the rows of the block table took a trip to memory more (1 M ray samples of four
// channels: scatter 52.7 -> 49.3 us, of both orders 55.6 -> 50.1, of the second 53.8 -> 50.1,
// as with the table's way alone; of five 68.7 -> 65.1, of eight 73.2 -> 68.3).  Kernels that
// gather as well use it before (and second order with grad_z, made to wait, 65 -> 92).
template <int N>
__device__ __forceinline__ void arrived(float (&v)[N]) {
#pragma unroll
    for (int k = 0; k < N; ++k) asm volatile("" : "+v"(v[k]));
}

// grad_emb[row[c], 0..E - 1] += part(c, v) of the eight corners for the lanes that are
// `on`; every lane of the wavefront must take part.  `runs`: find_runs of this tile.
template <int E, typename Part>
__device__ __forceinline__ void scatter_rows(LineAcc& acc, float* __restrict__ grad_emb,
                                             const uint32_t (&row)[8], bool on, const Runs& runs,
                                             Part part, int lane) {
    // (samples cells apart, scattered points: nothing to join)
    const bool want = on && (!runs.any || runs.tail);
    if (acc.aside) {
#pragma unroll
        for (int c = 0; c < 8; c += 2) {
            const uint32_t rows[2] = {row[c], row[c + 1]};
            float v[2][E];
            part(c, v[0]);
            part(c + 1, v[1]);
            if (runs.any) {
                sum_runs(runs, v[0]);
                sum_runs(runs, v[1]);
            }
            acc.send_two<E>(grad_emb, want, rows, v, lane);
        }
    } else {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            float v[E];
            part(c, v);
            if (runs.any) sum_runs(runs, v);
            acc.add<E>(grad_emb, want, row[c], v, lane);
        }
        acc.flush(grad_emb, lane);
    }
    acc.done();
}

__device__ __forceinline__ LineTable* line_table(unsigned char* smem, const QDev& a,
                                                 bool lds_lut, bool wanted) {
    if (!wanted) return nullptr;
    return reinterpret_cast<LineTable*>(smem + table_offset(a, 1, lds_lut)) +
           (threadIdx.x >> 6);
}

// Rows of E floats, by a lane each (16-byte aligned where E is four).
template <int E>
__device__ __forceinline__ void load_whole_row(const float* __restrict__ at, float (&v)[E]) {
    if constexpr (E == 4) {
        const float4 r = *reinterpret_cast<const float4*>(at);
        v[0] = r.x, v[1] = r.y, v[2] = r.z, v[3] = r.w;
    } else {
        const FloatRow<E> r = *reinterpret_cast<const FloatRow<E>*>(at);
#pragma unroll
        for (int k = 0; k < E; ++k) v[k] = r.v[k];
    }
}

template <int E>
__device__ __forceinline__ void load_row_once(const float* __restrict__ at, float (&v)[E]) {
    if constexpr (E == 4) {
        typedef float v4f __attribute__((ext_vector_type(4)));
        const v4f r = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(at));
        v[0] = r.x, v[1] = r.y, v[2] = r.z, v[3] = r.w;
    } else {
#pragma unroll
        for (int k = 0; k < E; ++k) v[k] = __builtin_nontemporal_load(at + k);
    }
}

template <int E>
__device__ __forceinline__ float row_product(const float (&a)[E], const float (&b)[E]) {
    if constexpr (E >= 8) {
        // pairs, pairs of pairs, ..., as a lane per channel adds them up: one after the
        // other, wide rows lose by the roundings of the sum what they gain by those of the
        // products (error against 64 bits, 2-norm: of eight channels 9.5e-8 and 9.7e-8, of
        // twelve 9.7e-8 and 1.03e-7; of five 9.3e-8 and 9.2e-8)
        constexpr int kWide = E > 8 ? 16 : 8;
        float p[kWide];
#pragma unroll
        for (int k = 0; k < kWide; ++k) p[k] = k < E ? __fmul_rn(a[k < E ? k : 0], b[k < E ? k : 0]) : 0.f;
#pragma unroll
        for (int n = kWide / 2; n > 0; n /= 2) {
#pragma unroll
            for (int k = 0; k < n; ++k) p[k] = __fadd_rn(p[2 * k], p[2 * k + 1]);
        }
        return p[0];
    } else {
        float dot = a[0] * b[0];
#pragma unroll
        for (int k = 1; k < E; ++k) dot += a[k] * b[k];
        return dot;
    }
}

// First-order backward, rows of E (formulas as in query_backward_forward_kernel).
template <int E, bool LDS, int OUT, int THREADS>
__global__ __launch_bounds__(THREADS, waves_of_rows(E, THREADS)) void
query_backward_forward_vec_kernel(
        QDev a, const float* __restrict__ z, float* __restrict__ grad_emb,
        float* __restrict__ grad_off, const float* __restrict__ gg_off,
        const float* __restrict__ z2) {
    extern __shared__ __align__(16) unsigned char smem[];
    const CellLut lut = stage_cell_lut<LDS, THREADS>(a, smem);
    const int lane = threadIdx.x & 63;
    const float* __restrict__ emb = static_cast<const float*>(a.emb);
    constexpr bool want_emb = (OUT & 1) != 0;
    constexpr bool want_off = (OUT & 2) != 0;
    constexpr bool second = (OUT & 4) != 0;
    LineAcc acc;
    acc.start(line_table(smem, a, LDS, want_emb), lane);
    const int64_t ntiles = (a.N + THREADS - 1) / THREADS;
    TileWalk walk(ntiles);
    for (int64_t tile = walk.next; tile < walk.end; tile += walk.step) {
        uint32_t row[8];
        float o[3];
        const int64_t q = tile * THREADS + threadIdx.x;
        const QueryInputs in = load_inputs(a, q);
        resolve_rows<LDS>(a, lut, in, row, o);
        const bool on = row[0] != kNoRow;
        float zq[E] = {}, yq[E] = {};
        float gg[3] = {0.f, 0.f, 0.f};
        if (on) {
            load_row_once<E>(z + q * E, zq);
            if constexpr (second) {
                load_row_once<E>(z2 + q * E, yq);
                gg[0] = __builtin_nontemporal_load(gg_off + q * 3 + 0) * static_cast<float>(a.offset_scale);
                gg[1] = __builtin_nontemporal_load(gg_off + q * 3 + 1) * static_cast<float>(a.offset_scale);
                gg[2] = __builtin_nontemporal_load(gg_off + q * 3 + 2) * static_cast<float>(a.offset_scale);
            }
        }
        AxisTerms<float> t;
        axis_terms<float, true>(o, a.smooth, t);
        // the gathered rows are used up before the scatter starts, which keeps
        // them out of the registers the scatter needs
        if constexpr (want_off) {
            float e[8][E];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
#pragma unroll
                for (int k = 0; k < E; ++k) e[c][k] = 0.f;
                if (on) load_whole_row<E>(emb + static_cast<int64_t>(row[c]) * E, e[c]);
            }
            float go[3] = {0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                float gw[3];
                corner_weight_grad<float>(t, c, gw);
                const float dot = row_product<E>(e[c], zq);
                go[0] += dot * gw[0];
                go[1] += dot * gw[1];
                go[2] += dot * gw[2];
            }
            if (q < a.N) {
                const float scale = static_cast<float>(a.offset_scale);
                __builtin_nontemporal_store(on ? go[0] * scale : 0.f, grad_off + q * 3 + 0);
                __builtin_nontemporal_store(on ? go[1] * scale : 0.f, grad_off + q * 3 + 1);
                __builtin_nontemporal_store(on ? go[2] * scale : 0.f, grad_off + q * 3 + 2);
            }
        }
        if constexpr (want_emb) {
            const Runs runs = find_runs(row[0], on, static_cast<uint32_t>(a.M), lane);
            acc.tile(runs.ordered, lane);
            if constexpr (!want_off) {
                arrived(zq);
                if constexpr (second) {
                    arrived(yq);
                    arrived(gg);
                }
            }
            SlopeTerms<float> slope;
            if constexpr (second) slope_terms<float>(t, gg, slope);
            scatter_rows<E>(acc, grad_emb, row, on, runs, [&](int c, float (&v)[E]) {
                const float w = corner_weight<float>(t, c);
#pragma unroll
                for (int k = 0; k < E; ++k) v[k] = w * zq[k];
                if constexpr (second) {
                    const float d = corner_slope<float>(t, slope, c);
#pragma unroll
                    for (int k = 0; k < E; ++k) v[k] += d * yq[k];
                }
            }, lane);
        }
    }
}

// Backward of the backward, rows of E (formulas as in
// query_backward_backward_kernel).
template <int E, bool LDS, int OUT, int THREADS>
__global__ __launch_bounds__(THREADS, waves_of_rows(E, THREADS)) void
query_backward_backward_vec_kernel(
        QDev a, const float* __restrict__ gg_off, const float* __restrict__ z,
        float* __restrict__ grad_z, float* __restrict__ grad_emb) {
    extern __shared__ __align__(16) unsigned char smem[];
    const CellLut lut = stage_cell_lut<LDS, THREADS>(a, smem);
    const int lane = threadIdx.x & 63;
    const float* __restrict__ emb = static_cast<const float*>(a.emb);
    constexpr bool want_emb = (OUT & 1) != 0;
    constexpr bool want_z = (OUT & 2) != 0;
    LineAcc acc;
    acc.start(line_table(smem, a, LDS, want_emb), lane);
    const int64_t ntiles = (a.N + THREADS - 1) / THREADS;
    TileWalk walk(ntiles);
    for (int64_t tile = walk.next; tile < walk.end; tile += walk.step) {
        uint32_t row[8];
        float o[3];
        const int64_t q = tile * THREADS + threadIdx.x;
        const QueryInputs in = load_inputs(a, q);
        resolve_rows<LDS>(a, lut, in, row, o);
        const bool on = row[0] != kNoRow;
        float zq[E] = {};
        float gg[3] = {0.f, 0.f, 0.f};
        if (on) {
            load_row_once<E>(z + q * E, zq);
            gg[0] = __builtin_nontemporal_load(gg_off + q * 3 + 0) * static_cast<float>(a.offset_scale);
            gg[1] = __builtin_nontemporal_load(gg_off + q * 3 + 1) * static_cast<float>(a.offset_scale);
            gg[2] = __builtin_nontemporal_load(gg_off + q * 3 + 2) * static_cast<float>(a.offset_scale);
        }
        AxisTerms<float> t;
        axis_terms<float, true>(o, a.smooth, t);
        if constexpr (want_z) {
            float e[8][E];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
#pragma unroll
                for (int k = 0; k < E; ++k) e[c][k] = 0.f;
                if (on) load_whole_row<E>(emb + static_cast<int64_t>(row[c]) * E, e[c]);
            }
            float gz[E] = {};
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                float gw[3];
                corner_weight_grad<float>(t, c, gw);
                const float d = gw[0] * gg[0] + gw[1] * gg[1] + gw[2] * gg[2];
#pragma unroll
                for (int k = 0; k < E; ++k) gz[k] += d * e[c][k];
            }
            if (q < a.N) {
                if constexpr (E == 4) {
                    typedef float v4f __attribute__((ext_vector_type(4)));
                    const v4f g4 = {on ? gz[0] : 0.f, on ? gz[1] : 0.f, on ? gz[2] : 0.f, on ? gz[3] : 0.f};
                    __builtin_nontemporal_store(g4, reinterpret_cast<v4f*>(grad_z + q * 4));
                } else if constexpr (E < 12 || want_emb) {
#pragma unroll
                    for (int k = 0; k < E; ++k) __builtin_nontemporal_store(on ? gz[k] : 0.f, grad_z + q * E + k);
                } else {
                    // (left to the caches, which join the pieces of a line: behind a scatter,
                    // 660 000 queries of twelve and sixteen channels in no order 107 -> 101 and
                    // 118 -> 100 us, by a lane per channel 100 and 98, in order 53 -> 50 and 74 ->
                    // 55; of eight, with two pieces, 120 -> 117, but in order 53.9 -> 56.6)
#pragma unroll
                    for (int k = 0; k < E; ++k) grad_z[q * E + k] = on ? gz[k] : 0.f;
                }
            }
        }
        if constexpr (want_emb) {
            const Runs runs = find_runs(row[0], on, static_cast<uint32_t>(a.M), lane);
            acc.tile(runs.ordered, lane);
            if constexpr (!want_z) {
                arrived(zq);
                arrived(gg);
            }
            scatter_rows<E>(acc, grad_emb, row, on, runs, [&](int c, float (&v)[E]) {
                float gw[3];
                corner_weight_grad<float>(t, c, gw);
                const float d = gw[0] * gg[0] + gw[1] * gg[1] + gw[2] * gg[2];
#pragma unroll
                for (int k = 0; k < E; ++k) v[k] = d * zq[k];
            }, lane);
        }
    }
}

// ---------------------------------------------------------------- host
size_t rows_smem(const QDev& d, int line_tables = 0) {
    return table_offset(d, 1, lut_in_lds(d)) + line_tables * sizeof(LineTable);
}

// Workgroups of the kernels with line tables (OUT bit 0) share one table of
// cells between eight wavefronts where two of them fit a CU (blocks of up to 576
// cells): 80 KB each and sixteen wavefronts on a CU, where three of 44 KB with
// four are twelve.  2^22 ray samples on 200 k blocks of 8^3: backward 221 -> 190
// us, second order 214 -> 187; 1.5 x 10^6 unordered queries 541 and 542 us as
// before (their rows leave past the tables, bound by requests).
// (Rows of twelve have registers for twelve wavefronts on a CU.)
constexpr int kWideRows = 8;
int vec_threads(const QDev& d, int out) {
    const bool wide = lut_in_lds(d) && (out & 1) != 0 && d.E <= kWideRows && 2 * rows_smem(d, 2 * kBlock / 64) <= kLdsPerCu;
    return wide ? 2 * kBlock : kBlock;
}

}  // namespace

template <int E>
int launch_bwd_fwd_vec(const QDev& d, const void* z, void* ge, void* go, const Second& also,
                       hipStream_t s) {
    const int out = gradients_wanted(ge, go, also);
    const int threads = vec_threads(d, out);
    const size_t smem = rows_smem(d, ge != nullptr ? threads / 64 : 0);
    const unsigned g = persistent_grid((d.N + threads - 1) / threads, smem, resident_rows(E, 1, out));
#define ASH_BF(L, O, T)                                                       \
    query_backward_forward_vec_kernel<E, L, O, T><<<g, T, smem, s>>>(    \
            d, static_cast<const float*>(z), static_cast<float*>(ge),         \
            static_cast<float*>(go), static_cast<const float*>(also.gg),      \
            static_cast<const float*>(also.z))
    if constexpr (E > 12) {
        if (lut_in_lds(d)) ASH_BF(true, 2, kBlock);
        else ASH_BF(false, 2, kBlock);
    } else if (E <= kWideRows && threads > kBlock) {
        constexpr int wide = E <= kWideRows ? 2 * kBlock : kBlock;   // (not built for others)
        if (out == 7) ASH_BF(true, 7, wide);
        else if (out == 5) ASH_BF(true, 5, wide);
        else if (out == 3) ASH_BF(true, 3, wide);
        else ASH_BF(true, 1, wide);
    } else if (lut_in_lds(d)) {
        if (out == 7) ASH_BF(true, 7, kBlock);
        else if (out == 5) ASH_BF(true, 5, kBlock);
        else if (out == 3) ASH_BF(true, 3, kBlock);
        else if (out == 1) ASH_BF(true, 1, kBlock);
        else if constexpr (E > 1) ASH_BF(true, 2, kBlock);
    } else {
        if (out == 7) ASH_BF(false, 7, kBlock);
        else if (out == 5) ASH_BF(false, 5, kBlock);
        else if (out == 3) ASH_BF(false, 3, kBlock);
        else if (out == 1) ASH_BF(false, 1, kBlock);
        else if constexpr (E > 1) ASH_BF(false, 2, kBlock);
    }
#undef ASH_BF
    ASH_LAUNCH_CHECK();
    return 0;
}

template <int E>
int launch_bwd_bwd_vec(const QDev& d, const void* gg, const void* z, void* gz,
                       void* ge, hipStream_t s) {
    const int out = (ge != nullptr ? 1 : 0) | (gz != nullptr ? 2 : 0);
    const int threads = vec_threads(d, out);
    const size_t smem = rows_smem(d, ge != nullptr ? threads / 64 : 0);
    const unsigned g = persistent_grid((d.N + threads - 1) / threads, smem, resident_rows(E, 2, out));
#define ASH_BB(L, O, T)                                                       \
    query_backward_backward_vec_kernel<E, L, O, T><<<g, T, smem, s>>>(   \
            d, static_cast<const float*>(gg), static_cast<const float*>(z),   \
            static_cast<float*>(gz), static_cast<float*>(ge))
    if constexpr (E > 12) {
        if (lut_in_lds(d)) ASH_BB(true, 2, kBlock);
        else ASH_BB(false, 2, kBlock);
    } else if (E <= kWideRows && threads > kBlock) {
        constexpr int wide = E <= kWideRows ? 2 * kBlock : kBlock;
        if (out == 3) ASH_BB(true, 3, wide);
        else ASH_BB(true, 1, wide);
    } else if (lut_in_lds(d)) {
        if (out == 3) ASH_BB(true, 3, kBlock);
        else if (out == 1) ASH_BB(true, 1, kBlock);
        else if constexpr (E > 1) ASH_BB(true, 2, kBlock);
    } else {
        if (out == 3) ASH_BB(false, 3, kBlock);
        else if (out == 1) ASH_BB(false, 1, kBlock);
        else if constexpr (E > 1) ASH_BB(false, 2, kBlock);
    }
#undef ASH_BB
    ASH_LAUNCH_CHECK();
    return 0;
}

template int launch_bwd_fwd_vec<ASH_ROW_WIDTH>(const QDev&, const void*, void*, void*, const Second&, hipStream_t);
template int launch_bwd_bwd_vec<ASH_ROW_WIDTH>(const QDev&, const void*, const void*, void*, void*, hipStream_t);

}  // namespace ash
