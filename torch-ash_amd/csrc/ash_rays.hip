// Rays through the active blocks of a grid (ash/src/sampler.cu:7-67 and
// :122-214): the near / far range of a ray and the samples inside blocks.
//
// Positions are origin + t * direction as a fused multiply-add (what nvcc makes
// of the reference's expression); the march is in cell units and a block is
// `grid2cell` cells wide.  Rays may come in world units: the kernels then bring
// them to cell units and their results back, operation by operation as torch
// evaluates `(x - origin) / cell_size` and `t * cell_size` on the device.
#include "ash_probe.h"

#include "../../include/ash_hip.h"

#include <cmath>
#include <type_traits>

namespace ash {
namespace {

constexpr int kBlock = 256;

// World units: cell units = (x - origin) * inv_cell, world = t * cell.  Neutral:
// origin null, inv_cell = cell = 1.
struct RayUnits {
    const float* origin;
    float inv_cell, cell;
};

__device__ __forceinline__ float to_cells(const RayUnits& u, float x, int axis) {
    const float o = u.origin != nullptr ? u.origin[axis] : 0.f;
    return __fmul_rn(__fsub_rn(x, o), u.inv_cell);
}

// Lane `l`'s value, and a condition that is the same in every lane.
__device__ __forceinline__ float lane_value(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ bool uniform(bool c) {
    return __builtin_amdgcn_readfirstlane(static_cast<int>(c)) != 0;
}

// A byte per block of the cube lo .. lo + edge - 1 (each axis), `mark` where the block
// is stored and anything else where it is not, in bricks of 4 x 4 x 8 blocks: a ray stays within a line of 128 for
// some eight steps.  With it a look-up is one load and fifteen instructions
// instead of the six loads and eighty of a bucket.  Behind the bytes stands a word
// that is `mark` if a block is stored outside: only then the table is asked about
// blocks out there (a ray that meets nothing is sampled far beyond its grid).
struct Volume {
    const uint8_t* at;   // null: none
    int32_t lo;
    uint32_t edge;
    uint32_t mark;       // 1 .. kMostMarks
};
constexpr uint32_t kMostMarks = ASH_RAY_VOLUME_MARKS;

// More than this does not stay in an XCD's L2.
constexpr int64_t kMaxVolume = int64_t{4} << 20;
// Making it takes two launches of 4 us each, which so many rays gain back: near
// and far of 3000 rays 15 -> 15 us, 4096 17 -> 14, 8192 29 -> 15, 32 768 79 -> 27;
// samples of 8000 rays 32 - 57 -> 36 - 48 (few blocks and short rays - many and
// long), 32 768 37 - 77 -> 38 - 55.
constexpr int64_t kVolumeRaysNearFar = 4096, kVolumeRaysSampling = 8192;
// One that is kept need not be cleared, which leaves one launch of 3 - 4 us, longer where
// the log is long.  Near and far, from the table -> with it, us: 1500 blocks, 1100 rays
// 10.7 -> 6.7, 4000 15.1 -> 6.9; 200 000 blocks 12.3 -> 8.4, 17.6 -> 9.0; 200 000 of 1.5 M in
// the log 1000 8.8 -> 9.2, 1500 11.1 -> 9.3; 1.2 M of 1.5 M 2500 14.0 -> 15.5.  Whole calls of
// samples, up to 16 | 32 | 64 | 128 of a ray: 2100 rays, 1500 blocks 27.3 -> 28.4 | 29.0 ->
// 29.7 | 31.2 -> 31.0 | 35.4 -> 33.3; 30 000 28.5 -> 28.9 | 31.2 -> 30.5 | 35.5 -> 33.0 | 40.1
// -> 36.1; 200 000 29.3 -> 29.2 | 33.3 -> 32.2 | 38.9 -> 35.2 | 46.9 -> 40.8; 8100 rays, 1500
// blocks 27.1 -> 28.5 | 29.5 -> 29.8 | 32.0 -> 31.4 | 36.3 -> 33.6: from 64 on they gain.
constexpr int64_t kKeptRaysNearFar = 1024, kKeptRaysSampling = 2048;
constexpr int64_t kKeptSamples = 64, kKeptLogPerRay = 384;

__host__ __device__ __forceinline__ int64_t volume_bytes(int64_t edge) {
    const int64_t flat = (edge + 3) / 4, tall = (edge + 7) / 8;
    return flat * flat * tall * 128;
}

constexpr int64_t kOutsideBytes = 16;   // of the word

// Bytes of a volume and its word, 0 where there is none.
int64_t volume_scratch(int lo, int hi) {
    const int64_t edge = static_cast<int64_t>(hi) - lo + 1;
    if (edge < 1 || edge > kMaxVolume) return 0;
    const int64_t bytes = volume_bytes(edge);
    return bytes <= kMaxVolume ? bytes + kOutsideBytes : 0;
}

// (to be asked for early and looked at late)
__device__ __forceinline__ uint32_t outside_word(const Volume& v) {
    return *reinterpret_cast<const uint32_t*>(v.at + volume_bytes(v.edge));
}

// (Of a block inside, no factor has more than 24 bits.)
__device__ __forceinline__ uint32_t volume_offset(const Volume& v, const uint32_t (&p)[3]) {
    const uint32_t flat = ((v.edge + 3) >> 2) & 0xffffu;
    // (the masks say so to the compiler: products of 32 bits take four times as long)
    const uint32_t slab = ((p[2] >> 3) & 0xffffu) * flat + (p[1] >> 2);
    const uint32_t brick = (slab & 0xffffffu) * flat + (p[0] >> 2);   // v_mad_u32_u24
    const uint32_t row = ((p[1] << 2) & ~3u) | (p[0] & 3u);
    const uint32_t place = ((p[2] << 4) & ~15u) | (row & 15u);
    return (brick << 7) | (place & 127u);
}

// The largest of a block's coordinates from the volume's first one (below `edge` of a
// block inside).
__device__ __forceinline__ uint32_t outermost(const uint32_t (&p)[3]) {
    const uint32_t xy = p[0] > p[1] ? p[0] : p[1];
    return xy > p[2] ? xy : p[2];
}

__device__ __forceinline__ bool in_volume(const Volume& v, const int32_t (&block)[3], uint32_t& at) {
    uint32_t p[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) p[a] = static_cast<uint32_t>(block[a]) - static_cast<uint32_t>(v.lo);
    at = volume_offset(v, p);
    return outermost(p) < v.edge;
}

__global__ __launch_bounds__(kBlock) void clear_volume_kernel(uint4* __restrict__ to, int64_t units) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i < units) to[i] = make_uint4(0u, 0u, 0u, 0u);
}

// Marks the stored blocks, from the log (keys of the general region, of which the
// log holds no code, lie outside every cube that fits).
__global__ __launch_bounds__(kBlock) void mark_volume_kernel(MapDev m, int identity, Volume v,
                                                             uint8_t* __restrict__ to) {
    const int64_t limit = identity ? static_cast<int64_t>(m.ctr[kCtrSize])
                                   : static_cast<int64_t>(m.capacity);
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    const uint64_t code = i < limit ? m.klog[i] : kEmpty;
    if (code == kEmpty) return;
    int32_t block[3];
    unpack_key<3>(code, block);
    uint32_t at;
    if (code < kTomb && in_volume(v, block, at)) {
        to[at] = static_cast<uint8_t>(v.mark);
    } else {
        *reinterpret_cast<uint32_t*>(to + volume_bytes(v.edge)) = v.mark;
    }
}

// Whether the blocks are stored, every lane for itself: K look-ups per lane, none
// in a branch, so that all are on their way together; the table is asked only if a
// block lies outside the volume.
template <int K>
__device__ __forceinline__ void are_stored(const MapDev& m, const Volume& v, const int32_t (&block)[K][3],
                                           const bool (&active)[K], bool (&stored)[K]) {
    bool inside[K], others = false;
    uint8_t word[K];
#pragma unroll
    for (int h = 0; h < K; ++h) {
        uint32_t at;
        inside[h] = in_volume(v, block[h], at) & active[h];
        word[h] = v.at[inside[h] ? at : 0u];
        others = others | (active[h] & !inside[h]);
    }
#pragma unroll
    for (int h = 0; h < K; ++h) stored[h] = inside[h] & (word[h] == v.mark);
    if (__ballot(others) != 0) {
#pragma unroll
        for (int h = 0; h < K; ++h) {
            int32_t idx;
            stored[h] = stored[h] | find_key_alone<3>(m, block[h], active[h] & !inside[h], idx);
        }
    }
}

// floor, in one instruction: what a conversion of floorf(x) gives, for all x but those
// that are not a number.
__device__ __forceinline__ int32_t floor_to_int(float x) {
    int32_t r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

__device__ __forceinline__ void ray_block(const float (&o)[3], const float (&d)[3],
                                          float t, float cell2grid,
                                          int32_t (&block)[3], float (&x)[3]) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        x[a] = fmaf(t, d[a], o[a]);
        block[a] = static_cast<int32_t>(floorf(__fmul_rn(x[a], cell2grid)));
    }
}

// The same from the table; the first lane of a run of equal blocks asks.
__device__ __forceinline__ bool is_stored_by_runs(const MapDev& m, const int32_t (&block)[3], bool active) {
    const int lane = threadIdx.x & 63;
    // (asked of every lane: of one that takes no part, the shift gives back the asker's own)
    const int32_t active_before = lane_before(static_cast<int32_t>(active));
    int same = lane > 0 && active && active_before != 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) same &= lane_before(block[a]) == block[a];
    int32_t idx;
    const bool asked = find_key_alone<3>(m, block, active && !same, idx);
    const uint64_t heads = __ballot(!same);
    return __shfl(static_cast<int>(asked), 63 - __builtin_clzll(heads & (~0ull >> (63 - lane)))) != 0;
}

// One wavefront per ray: the march of ray_find_near_far visits the parameters
// t_0 = t_min, t_{k+1} = t_k + step regardless of what it finds, so lane l of
// round r takes step 64 r + l, the 64 look-ups go out together, and the near /
// far recurrence is then replayed over the hits in step order.  The march ends
// at the first step that is at or beyond t_max or outside the box, exactly where
// the sequential loop stops.
//
// The parameters are the same for every ray, so the host works the chain of
// additions out (the same IEEE additions) for the first kChain steps and hands it
// over with the launch, 64 additions per round less; and the recurrence takes
// `far` from the last hit and `near`, once it is set, only from the number of hits:
// all its subtractions at once where they are exact (Exact::near_below), else one
// after the other (two instructions each).
constexpr int kChain = 512;

struct StepChain {
    float t[kChain];
};

// What floats hold without rounding, as the host finds it: `near`, as long as it is
// not negative, minus any number of steps if `near` is at most near_below (both are
// then whole multiples of the last place of `near`), and, with `steps`, the
// parameter of every step up to the first at or beyond t_max, t_min + k * step.
struct Exact {
    float near_below;
    bool steps;
};

template <bool VOLUME>
__global__ __launch_bounds__(kBlock) void ray_near_far_kernel(
        MapDev m, Volume volume, const float* __restrict__ origins,
        const float* __restrict__ directions, RayUnits u, const float* __restrict__ bbox_min,
        const float* __restrict__ bbox_max, int64_t n, float t_min, float t_max,
        float grid2cell, float* __restrict__ nears, float* __restrict__ fars, Exact exact, StepChain chain) {
    const int lane = threadIdx.x & 63;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * (kBlock / 64) + (threadIdx.x >> 6);
    if (i >= n) return;  // whole wavefronts leave together
    const float cell2grid = static_cast<float>(1.0 / grid2cell);
    const float t_grid_step = static_cast<float>(grid2cell * 0.5);
    float o[3], d[3], lo[3], hi[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        o[a] = to_cells(u, origins[i * 3 + a], a);
        d[a] = directions[i * 3 + a];
        lo[a] = to_cells(u, bbox_min[a], a);
        hi[a] = to_cells(u, bbox_max[a], a);
    }
    float near = -1.f, far = t_max;
    float t = 0.f;
    for (int first = 0;; first += 64) {
        if (first < kChain) {
            t = chain.t[first + lane];
        } else {
            for (int j = 0; j < 64; ++j) t += t_grid_step;
        }
        int32_t block[1][3];
        float x[3];
        ray_block(o, d, t, cell2grid, block[0], x);
        bool go = t < t_max;
#pragma unroll
        for (int a = 0; a < 3; ++a) go = go && x[a] >= lo[a] && x[a] <= hi[a];
        const uint64_t stop = __ballot(!go);
        const int first_stop = stop ? __builtin_ctzll(stop) : 64;
        const bool active[1] = {lane < first_stop};
        bool found[1];
        if constexpr (VOLUME) {
            are_stored(m, volume, block, active, found);
        } else {
            // (steps are half a block apart: neighbouring lanes often stand in the
            // same block and share a look-up)
            int32_t idx;
            found[0] = find_block_by_runs(m, block[0], active[0], idx);
        }
        uint64_t hits = __ballot(found[0] && active[0]);
        if (hits) {
            far = fminf(lane_value(t, 63 - __builtin_clzll(hits)) + t_grid_step, t_max);
            if (t_min >= 0.f) {   // near never turns negative again
                int steps = __popcll(hits);
                if (uniform(near < 0.f)) {
                    near = lane_value(t, __builtin_ctzll(hits));
                    --steps;
                }
                if (uniform(near <= exact.near_below)) {
                    near = fmaxf(fmaf(static_cast<float>(-steps), t_grid_step, near), t_min);
                } else {
                    for (; steps > 0; --steps) near = fmaxf(near - t_grid_step, t_min);
                }
            } else {
                while (hits) {
                    const float t_hit = lane_value(t, __builtin_ctzll(hits));
                    near = near < 0.f ? t_hit : fmaxf(near - t_grid_step, t_min);
                    hits &= hits - 1;
                }
            }
        }
        if (first_stop < 64) break;
    }
    if (lane == 0) {
        nears[i] = __fmul_rn(near, u.cell);
        fars[i] = __fmul_rn(far, u.cell);
    }
}

// The same march for two rays per wavefront, lane j of a ray on steps 32 h + j:
// where the recurrence is exact and a volume stands, t_min is not negative and the
// parameters are at hand (exact, or all in the chain).  A ray then needs no more
// than its first and its last hit and their number, and half as many wavefronts wait
// for their rays' words.
//
// Positions do not turn back along an axis (their roundings keep the order), so that a
// ray inside the box at its first step stays inside until one step from which on it is
// outside.  That step, the ray's end, is looked for first, 32 steps about where the
// division puts it, and if it is not among them by intervals of 32 parts; the steps
// before it are then only looked up, without the box.
//
// Bound by vector instructions (410 of a wavefront): with the box asked at every step
// 22.4 us for 32 768 rays across 200 000 blocks, 15.5 with the end found first; of rays with
// one component of zero 20.5 and 14.4 (16.3 where such a component sent the first guess to
// the ray's start).
struct RaySteps {
    int most;         // whose parameter lies below t_max
    float per_step;   // about 1 / step, for the first guess
};

template <bool EXACT>   // Exact::steps
__global__ __launch_bounds__(kBlock) void ray_near_far_pairs_kernel(
        MapDev m, Volume volume, const float* __restrict__ origins,
        const float* __restrict__ directions, RayUnits u, const float* __restrict__ bbox_min,
        const float* __restrict__ bbox_max, int64_t n, float t_min, float t_max,
        float grid2cell, float cell2grid, float* __restrict__ nears, float* __restrict__ fars, RaySteps steps, StepChain chain) {
    const int lane = threadIdx.x & 63;
    const int j = lane & 31, shift = lane & 32;
    const int64_t pair = static_cast<int64_t>(blockIdx.x) * (kBlock / 64) +
                         __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (2 * pair >= n) return;  // whole wavefronts leave together
    const int64_t i = 2 * pair + (shift >> 5);
    const int32_t from = i < n ? 3 * (shift >> 5) : 0;
    const float* const o_from = origins + 6 * pair;
    const float* const d_from = directions + 6 * pair;
    const float t_grid_step = static_cast<float>(grid2cell * 0.5);
    const uint32_t outside = outside_word(volume);
    float o[3], d[3], lo[3], hi[3], zero[3] = {0.f, 0.f, 0.f};
    if (u.origin != nullptr) {
#pragma unroll
        for (int a = 0; a < 3; ++a) zero[a] = u.origin[a];
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        auto cells = [&](float x) { return __fmul_rn(__fsub_rn(x, zero[a]), u.inv_cell); };
        o[a] = cells(o_from[from + a]);
        d[a] = d_from[from + a];
        lo[a] = cells(bbox_min[a]);
        hi[a] = cells(bbox_max[a]);
    }
    // (any k >= 0; beyond the chain the last of its parameters, a step nobody takes)
    auto parameter = [&](int k) {
        return EXACT ? fmaf(static_cast<float>(k), t_grid_step, t_min)
                     : chain.t[k < kChain ? k : kChain - 1];
    };
    auto inside = [&](int k) {
        const float t = parameter(k);
        bool in = k < steps.most;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const float x = fmaf(t, d[a], o[a]);
            in = in & (x >= lo[a]) & (x <= hi[a]);
        }
        return in;
    };
    auto of_ray = [&](bool c) {   // its lanes' conditions
        const uint64_t all = __builtin_amdgcn_ballot_w64(c);
        return shift != 0 ? static_cast<uint32_t>(all >> 32) : static_cast<uint32_t>(all);
    };

    // the ray's end: above `low`, which is inside, and at most `high`
    int low = 0, high = inside(0) ? steps.most : 0;
    {
        float at = t_max;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            // (by the sign bit: a component of +0 or -0 gives +infinity, and 0 * infinity,
            // which is no number, does not count)
            const float side = __float_as_int(d[a]) >= 0 ? hi[a] : lo[a];
            at = fminf(at, (side - o[a]) * __builtin_amdgcn_rcpf(d[a]));
        }
        const float guess = fminf(fmaxf((at - t_min) * steps.per_step - 16.f, 0.f), static_cast<float>(steps.most));
        const int base = static_cast<int>(guess);
        const uint32_t in = of_ray(high > 0 && inside(base + j));
        if (in != 0u) {
            low = base + 31 - __clz(in);
            if (in != ~0u) high = low + 1;
        } else if (high > base && base > 0) {
            high = base;
        }
    }
    while (__ballot(high - low > 1) != 0) {
        const int part = (high - low + 31) >> 5;   // (at least one, and less than high - low)
        const int k = low + (j + 1) * part;
        const int in = __popc(of_ray(k < high && inside(k)));
        const int above = low + (in + 1) * part;
        if (high - low > 1) {
            high = above < high ? above : high;
            low += in * part;
        }
    }
    const int end = i < n ? high : 0;

    int hits[2] = {0, 0}, first_hit[2] = {0, 0}, last_hit[2] = {0, 0};
    auto count = [&](uint64_t stands, int first) {
        const int words[2] = {static_cast<int>(stands), static_cast<int>(stands >> 32)};
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            // (scalar, also the test for zero of the upper half)
            const auto word = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(words[r]));
            if (word == 0u) continue;
            if (hits[r] == 0) first_hit[r] = first + __builtin_ctz(word);
            last_hit[r] = first + 31 - __builtin_clz(word);
            hits[r] += __builtin_popcount(word);
        }
    };
    const int ends[2] = {__builtin_amdgcn_readlane(end, 0), __builtin_amdgcn_readlane(end, 32)};
    const int most = ends[0] > ends[1] ? ends[0] : ends[1];
    if (uniform(outside != volume.mark)) {
        // (exact parameters are also the sums of these steps, and in their order)
        float t = parameter(j);
        const float t_end = parameter(end);
        const auto last_byte = static_cast<uint32_t>(volume_bytes(volume.edge) - 1);
        auto round = [&](int first, auto looks) {
            constexpr int kLooks = decltype(looks)::value;
            uint8_t word[kLooks];
            uint64_t before[kLooks];
#pragma unroll
            for (int h = 0; h < kLooks; ++h) {
                if constexpr (EXACT) {
                    before[h] = __builtin_amdgcn_ballot_w64(t < t_end);
                } else {
                    t = parameter(first + 32 * h + j);
                    before[h] = __builtin_amdgcn_ballot_w64(first + 32 * h + j < end);
                }
                uint32_t p[3];
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    p[a] = static_cast<uint32_t>(floor_to_int(__fmul_rn(fmaf(t, d[a], o[a]), cell2grid))) -
                           static_cast<uint32_t>(volume.lo);
                }
                // (outside: anywhere)
                const uint32_t at = volume_offset(volume, p);
                word[h] = volume.at[at < last_byte ? at : last_byte];
                before[h] &= __builtin_amdgcn_ballot_w64(outermost(p) < volume.edge);
                if constexpr (EXACT) t += 32.f * t_grid_step;
            }
            __builtin_amdgcn_sched_barrier(0);   // (all are on their way before one is waited for)
#pragma unroll
            for (int h = 0; h < kLooks; ++h) {
                count(before[h] & __builtin_amdgcn_ballot_w64(word[h] == volume.mark), first + 32 * h);
            }
        };
        int first = 0;
        for (; most - first > 64; first += 128) round(first, std::integral_constant<int, 4>());
        if (most - first > 32) {
            round(first, std::integral_constant<int, 2>());
        } else if (most > first) {
            round(first, std::integral_constant<int, 1>());
        }
    } else {
        for (int first = 0; first < most; first += 64) {
            int32_t block[2][3];
            float x[3];
            bool active[2], found[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int k = first + 32 * h + j;
                ray_block(o, d, parameter(k), cell2grid, block[h], x);
                active[h] = k < end;
            }
            are_stored(m, volume, block, active, found);
#pragma unroll
            for (int h = 0; h < 2; ++h) count(__builtin_amdgcn_ballot_w64(found[h]), first + 32 * h);
        }
    }
    if (j == 0 && i < n) {
        float near = -1.f, far = t_max;
        const int met = shift != 0 ? hits[1] : hits[0];
        if (met > 0) {
            near = fmaxf(fmaf(static_cast<float>(1 - met), t_grid_step,
                              parameter(shift != 0 ? first_hit[1] : first_hit[0])), t_min);
            far = fminf(parameter(shift != 0 ? last_hit[1] : last_hit[0]) + t_grid_step, t_max);
        }
        nears[i] = __fmul_rn(near, u.cell);
        fars[i] = __fmul_rn(far, u.cell);
    }
}

// The march of ray_sample.  counts != nullptr: allocation pass; otherwise the
// assignment pass, which writes the samples of ray i at prefix[i - 1] ..
// prefix[i].  An allocation pass with `stage` also keeps the first `stride`
// samples of ray i as pairs (t_near, t_far) at stage[i * stride + k], so that
// the assignment pass can be a copy instead of a second march; with `groups` it
// leaves the sum and the largest of its workgroup's counts there.
//
// The reference looks the block under t up at every step, one dependent look-up
// after the other.  What it does next depends on one bit only, though, so the
// LPR lanes of a ray stand on the next LPR positions of the march as it goes on
// if all of them are stored (or all are not: whichever the latest one was), look
// them up at once, and the march takes as many of these steps as turn out that
// way, and the first one that does not.  (32 768 rays of 31 samples in 200 000
// blocks: 113 us when the eight lanes looked blocks up ahead and a step went by
// whether one of them held the block under t, 55 with these runs; 23.5 from the volume,
// 20.1 with a ray's numbers asked for together, its steps worked out as masks by the
// scalar unit and no block outside asked for.  What bounds it now is the chain of
// rounds: a wavefront takes as many as the longest of its eight rays, 17 on average.)
struct GroupSamples {
    int64_t sum, most;
};

template <int LPR, bool VOLUME>
__global__ __launch_bounds__(kBlock) void ray_sample_kernel(
        MapDev m, Volume volume, const float* __restrict__ origins,
        const float* __restrict__ directions, RayUnits u, const float* __restrict__ ray_nears,
        const float* __restrict__ ray_fars, float near_for_all, float far_for_all, int64_t n,
        float max_samples, float grid2cell, int64_t* __restrict__ counts,
        const int64_t* __restrict__ prefix, int64_t* __restrict__ ray_indices,
        float* __restrict__ t_nears, float* __restrict__ t_fars,
        float2* __restrict__ stage, int64_t stride, GroupSamples* __restrict__ groups) {
    const int lane = threadIdx.x & 63;
    const int64_t gid = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    const int64_t i = gid / LPR;
    const int j = static_cast<int>(gid % LPR);
    const bool writer = j == 0;   // the lane of a ray that stores its results
    const bool active = i < n;
    const float cell2grid = static_cast<float>(1.0 / grid2cell);
    // (nothing under a condition of the lane's, so that all of a ray is on its way at once)
    const int64_t from = active ? i : n - 1;
    float o[3], d[3], zero[3] = {0.f, 0.f, 0.f};
    float ray_near = near_for_all, ray_far = far_for_all;
    uint32_t beyond = 0;
    if constexpr (VOLUME) beyond = outside_word(volume);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        o[a] = origins[from * 3 + a];
        d[a] = directions[from * 3 + a];
    }
    if (ray_nears != nullptr) ray_near = ray_nears[from];
    if (ray_fars != nullptr) ray_far = ray_fars[from];
    if (u.origin != nullptr) {
#pragma unroll
        for (int a = 0; a < 3; ++a) zero[a] = u.origin[a];
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) o[a] = __fmul_rn(__fsub_rn(o[a], zero[a]), u.inv_cell);
    if (ray_nears != nullptr) ray_near = __fmul_rn(ray_near, u.inv_cell);
    if (ray_fars != nullptr) ray_far = __fmul_rn(ray_far, u.inv_cell);
    const float t_step = fmaxf(0.7f, __fdiv_rn(ray_far - ray_near, max_samples));
    const float t_grid_step = __fmul_rn(t_step, grid2cell);
    const int64_t start = (counts == nullptr && active && i > 0) ? prefix[i - 1] : 0;
    float2* const staged = stage != nullptr ? stage + i * stride : nullptr;
    float t = ray_near, t_near = ray_near;
    // (a march has less than 2^26 steps: each is 0.7 or more, and it ends where one no
    // longer advances t)
    int32_t local = 0;
    bool live = active && t < ray_far && t > -INFINITY;
    auto keep = [&](int32_t k, float from, float to) {
        if (counts == nullptr) {
            ray_indices[start + k] = i;
            t_nears[start + k] = from;
            t_fars[start + k] = to;
        } else if (stage != nullptr && k < stride) {
            staged[k] = make_float2(from, to);
        }
    };
    // What a position's block is taken from its three coordinates in one instruction
    // each, which a ray that has no finite origin and direction does not allow.
    bool outside = false, odd = false;
    uint32_t last_byte = 0;
    if constexpr (VOLUME) {
        outside = uniform(beyond == volume.mark);
        odd = !(fabsf(o[0]) + fabsf(o[1]) + fabsf(o[2]) + fabsf(d[0]) + fabsf(d[1]) + fabsf(d[2]) < INFINITY);
        last_byte = static_cast<uint32_t>(volume_bytes(volume.edge) - 1);
    }
    // What the lanes find is a mask, and all rays' steps are worked out of masks at
    // once, by the scalar unit: a bit per lane, LPR bits per ray.
    const int shift = lane & ~(LPR - 1);
    constexpr uint64_t kFirst = LPR == 8 ? 0x0101010101010101ull : 0x1111111111111111ull;
    constexpr uint64_t kLast = kFirst << (LPR - 1);
    auto of_ray = [&](uint64_t mask) {
        const uint32_t half = shift >= 32 ? static_cast<uint32_t>(mask >> 32) : static_cast<uint32_t>(mask);
        return (half >> (shift & 31)) & ((1u << LPR) - 1u);
    };
    bool run_stored = true;   // what the positions ahead are taken for
    while (__builtin_amdgcn_ballot_w64(live) != 0) {
        const float by = run_stored ? t_step : t_grid_step;
        float at = t;
#pragma unroll
        for (int k = 1; k < LPR; ++k) at = j >= k ? at + by : at;
        const float next = at + by;
        // (a step that no longer advances t -- range far beyond fp32 resolution --
        // would never end; the reference has no such guard)
        const uint64_t forward = __builtin_amdgcn_ballot_w64(next > at);
        const uint64_t stands = __builtin_amdgcn_ballot_w64(live & (at < ray_far)) & ((forward << 1) | kFirst);
        uint64_t stored;
        bool general = !VOLUME;
        if constexpr (VOLUME) general = outside || __builtin_amdgcn_ballot_w64(live & odd) != 0;
        if (general) {
            const bool asks[1] = {__builtin_amdgcn_inverse_ballot_w64(stands)};
            int32_t block[1][3];
            float x[3];
            ray_block(o, d, at, cell2grid, block[0], x);
            bool found[1];
            if constexpr (VOLUME) {
                are_stored(m, volume, block, asks, found);
            } else {
                found[0] = is_stored_by_runs(m, block[0], asks[0]);
            }
            stored = __builtin_amdgcn_ballot_w64(found[0]);
        } else {
            uint32_t p[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                p[a] = static_cast<uint32_t>(floor_to_int(__fmul_rn(fmaf(at, d[a], o[a]), cell2grid))) -
                       static_cast<uint32_t>(volume.lo);
            }
            // (outside: anywhere)
            const uint32_t where = volume_offset(volume, p);
            stored = __builtin_amdgcn_ballot_w64(outermost(p) < volume.edge) &
                     __builtin_amdgcn_ballot_w64(volume.at[where < last_byte ? where : last_byte] == volume.mark);
        }
        const uint64_t expected = stands & ~(stored ^ __builtin_amdgcn_ballot_w64(run_stored));
        // a ray takes its steps up to the first that is not as expected: the ones at the
        // lower end of its bits, by a carry that its last bit stops
        const uint64_t low = expected & ~kLast, carried = low + kFirst;
        const uint64_t taken = (low & ~carried) | (expected & carried & kLast);
        const uint64_t turns = carried & ~low & ~taken & stands;   // there it stands on the other kind
        const int run = __popc(of_ray(taken));
        const bool turn = of_ray(turns) != 0;
        const float behind = __shfl(next, shift + run - 1);
        const float reached = run > 0 ? behind : t;
        t = reached;
        bool on = t < ray_far;
        if ((taken & ~forward) != 0) on = on && of_ray(taken & ~forward) == 0;
        const float turned = t + (run_stored ? t_grid_step : t_step);
        if (turn) {
            on = turned < ray_far && turned > t;
            t = turned;
        }
        const int more = run_stored ? run : (turn ? 1 : 0);   // samples
        if (j < more) keep(local + j, j > 0 ? at : t_near, run_stored ? next : t);
        local += more;
        if (more > 0) t_near = run_stored ? reached : t;
        run_stored = run_stored != turn;
        live = live && on;
    }
    if (active && writer && counts != nullptr) counts[i] = local;
    if (groups != nullptr) {
        // (the writers are LPR lanes apart)
        int32_t sum = active && writer ? local : 0, most = sum;
#pragma unroll
        for (int b = 32; b >= LPR; b >>= 1) {
            sum += __shfl_xor(sum, b);
            const int32_t other = __shfl_xor(most, b);
            most = other > most ? other : most;
        }
        __shared__ GroupSamples s_wave[kBlock / 64];
        if (lane == 0) s_wave[threadIdx.x >> 6] = {sum, most};
        __syncthreads();
        if (threadIdx.x == 0) {
            GroupSamples g = s_wave[0];
#pragma unroll
            for (int w = 1; w < kBlock / 64; ++w) {
                g.sum += s_wave[w].sum;
                g.most = s_wave[w].most > g.most ? s_wave[w].most : g.most;
            }
            groups[blockIdx.x] = g;
        }
    }
}

// One workgroup turns the sums of the march's workgroups into running sums (what
// lies before each, in place) and leaves the number of samples and the largest
// count of a ray for the host.
constexpr int kScanThreads = 1024;

__global__ __launch_bounds__(kScanThreads) void ray_scan_kernel(GroupSamples* __restrict__ groups,
                                                                int n, uint64_t* landing,
                                                                int32_t stamp) {
    __shared__ int64_t s_sum[kScanThreads / 64];
    __shared__ int64_t s_most[kScanThreads / 64];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int per = (n + kScanThreads - 1) / kScanThreads;
    const int first = threadIdx.x * per;
    const int last = first + per < n ? first + per : n;
    int64_t sum = 0, most = 0;
    for (int g = first; g < last; ++g) {
        sum += groups[g].sum;
        most = groups[g].most > most ? groups[g].most : most;
    }
    int64_t incl = sum;
#pragma unroll
    for (int b = 1; b < 64; b <<= 1) {
        const int64_t up = __shfl_up(incl, b);
        if (lane >= b) incl += up;
        const int64_t other = __shfl_xor(most, b);
        most = other > most ? other : most;
    }
    if (lane == 63) s_sum[wave] = incl;
    if (lane == 0) s_most[wave] = most;
    __syncthreads();
    int64_t before = incl - sum, total = 0;
    for (int w = 0; w < kScanThreads / 64; ++w) {
        if (w < wave) before += s_sum[w];
        total += s_sum[w];
        most = s_most[w] > most ? s_most[w] : most;
    }
    if (threadIdx.x == 0) {
        const int32_t words[4] = {static_cast<int32_t>(total), static_cast<int32_t>(total >> 32),
                                  static_cast<int32_t>(most), static_cast<int32_t>(most >> 32)};
#pragma unroll
        for (int w = 0; w < 4; ++w) leave_word(landing + w, words[w], stamp);
    }
    if (per == 1) {
        if (first < last) groups[first].sum = before;
        return;
    }
    for (int g = first; g < last; ++g) {
        const int64_t own = groups[g].sum;
        groups[g].sum = before;
        before += own;
    }
}

// The staged samples of `rays` rays, the share of one workgroup of the march,
// copied to their place.  Also the running sums of the counts.  Bound by its waits for
// memory: four samples of a thread are on their way together, and none of its lanes waits
// for a longer ray (eight lanes per ray, a sample at a time: 32 768 rays, a million samples,
// 10.7 -> 8.5 us; 100 000 rays of up to 128 with all their launches 149 -> 141).
constexpr int kAtOnce = 4;
constexpr int kMostRays = kBlock / 4;   // of a workgroup, a power of two (lanes_per_ray)

__global__ __launch_bounds__(kBlock) void ray_place_kernel(
        const int64_t* __restrict__ counts, const GroupSamples* __restrict__ groups,
        const float2* __restrict__ stage, int64_t stride, int64_t n, int rays, float cell,
        int64_t* __restrict__ ray_indices, float* __restrict__ t_nears,
        float* __restrict__ t_fars, int64_t* __restrict__ prefix) {
    __shared__ int64_t s_incl[kBlock];
    __shared__ int64_t s_wave[kBlock / 64];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int64_t first = static_cast<int64_t>(blockIdx.x) * rays;
    const int64_t own = tid < rays && first + tid < n ? counts[first + tid] : 0;
    const int64_t start = groups[blockIdx.x].sum;
    int64_t incl = own;
#pragma unroll
    for (int b = 1; b < 64; b <<= 1) {
        const int64_t up = __shfl_up(incl, b);
        if (lane >= b) incl += up;
    }
    if (lane == 63) s_wave[tid >> 6] = incl;
    __syncthreads();
    incl += start;
    for (int w = 0; w < (tid >> 6); ++w) incl += s_wave[w];
    s_incl[tid] = incl;
    if (tid < rays && first + tid < n) prefix[first + tid] = incl;
    __syncthreads();
    // consecutive threads, consecutive samples, whichever ray they belong to
    const int64_t total = s_incl[kBlock - 1] - start;
    for (int64_t t = tid; t < total; t += kBlock * kAtOnce) {
        int ray[kAtOnce];
        float2 s[kAtOnce];
#pragma unroll
        for (int h = 0; h < kAtOnce; ++h) {
            const int64_t at = start + (t + kBlock * h < total ? t + kBlock * h : t);
            int r = 0;   // rays that end at or before the sample
#pragma unroll
            for (int step = kMostRays / 2; step > 0; step >>= 1) {
                if (s_incl[r + step - 1] <= at) r += step;
            }
            ray[h] = r;
            s[h] = stage[(first + r) * stride + at - (r > 0 ? s_incl[r - 1] : start)];
        }
#pragma unroll
        for (int h = 0; h < kAtOnce; ++h) {
            if (t + kBlock * h >= total) break;
            const int64_t at = start + t + kBlock * h;
            ray_indices[at] = first + ray[h];
            t_nears[at] = __fmul_rn(s[h].x, cell);
            t_fars[at] = __fmul_rn(s[h].y, cell);
        }
    }
}

// Assignment pass from the staged samples and running sums of the caller's: one
// thread per staged slot.
__global__ __launch_bounds__(kBlock) void ray_compact_kernel(
        const int64_t* __restrict__ counts, const int64_t* __restrict__ prefix,
        const float2* __restrict__ stage, int64_t stride, int64_t n,
        int64_t* __restrict__ ray_indices, float* __restrict__ t_nears,
        float* __restrict__ t_fars) {
    const int64_t slot = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (slot >= n * stride) return;
    const int64_t i = slot / stride;
    const int64_t k = slot - i * stride;
    if (k >= counts[i]) return;
    const int64_t out = (i > 0 ? prefix[i - 1] : 0) + k;
    const float2 s = stage[slot];
    ray_indices[out] = i;
    t_nears[out] = s.x;
    t_fars[out] = s.y;
}

// Lanes per ray of the sampling march: eight, and four where there are rays
// enough that the positions looked up in vain weigh more than the rounds (100 000
// rays of up to 32 / 128 samples: 57 / 96 us and 46 / 90; 8000 rays: 39 / 48 and
// 39 / 55).
constexpr int64_t kFewLanesFrom = int64_t{1} << 16;

int lanes_per_ray(int64_t n) { return n < kFewLanesFrom ? 8 : 4; }

unsigned march_groups(int64_t n) {
    return static_cast<unsigned>((n * lanes_per_ray(n) + kBlock - 1) / kBlock);
}

struct March {
    const float *origins, *directions;
    RayUnits units;
    const float *nears, *fars;
    float near_for_all, far_for_all;
    int64_t n;
    float max_samples, grid2cell;
};

int launch_march(ash_map_t* map, const Volume& volume, const March& r, int64_t* counts, const int64_t* prefix,
                 int64_t* ray_indices, float* t_nears, float* t_fars, float* stage, int64_t stride,
                 GroupSamples* groups, hipStream_t s) {
    const bool eight = lanes_per_ray(r.n) == 8;
    auto kernel = volume.at != nullptr
                          ? (eight ? ray_sample_kernel<8, true> : ray_sample_kernel<4, true>)
                          : (eight ? ray_sample_kernel<8, false> : ray_sample_kernel<4, false>);
    kernel<<<march_groups(r.n), kBlock, 0, s>>>(
            map->d, volume, r.origins, r.directions, r.units, r.nears, r.fars, r.near_for_all, r.far_for_all,
            r.n, r.max_samples, r.grid2cell, counts, prefix, ray_indices, t_nears, t_fars,
            reinterpret_cast<float2*>(stage), stride, groups);
    ASH_LAUNCH_CHECK();
    return 0;
}

// The volume of the map's blocks in lo .. hi, if there is room for one.  `mark` 0: its
// bytes hold anything and are cleared; else none of them holds `mark`.  (A call that
// clears launches one kernel more, 3 - 4 us.)
int make_volume(ash_map_t* map, uint8_t* bytes, int lo, int hi, int mark, Volume& v, hipStream_t s) {
    v = {};
    if (bytes == nullptr) return 0;
    if (mark < 0 || mark > static_cast<int>(kMostMarks)) ASH_FAIL("rays: a volume's mark must be 0 .. 255");
    const int64_t edge = static_cast<int64_t>(hi) - lo + 1;
    if (edge < 1 || volume_bytes(edge) > kMaxVolume) ASH_FAIL("rays: too many blocks for a volume");
    if (reinterpret_cast<uintptr_t>(bytes) % 16 != 0) ASH_FAIL("rays: the volume must be 16-byte aligned");
    v = {bytes, lo, static_cast<uint32_t>(edge), static_cast<uint32_t>(mark)};
    if (mark == 0) {
        v.mark = 1;
        const int64_t units = (volume_bytes(edge) + kOutsideBytes) / 16;
        clear_volume_kernel<<<static_cast<unsigned>((units + kBlock - 1) / kBlock), kBlock, 0, s>>>(
                reinterpret_cast<uint4*>(bytes), units);
        ASH_LAUNCH_CHECK();
    }
    mark_volume_kernel<<<static_cast<unsigned>((map->capacity + kBlock - 1) / kBlock), kBlock, 0, s>>>(
            map->d, heap_in_order(map) ? 1 : 0, v, bytes);
    ASH_LAUNCH_CHECK();
    return 0;
}

constexpr RayUnits kCellUnits = {nullptr, 1.f, 1.f};

int check_rays(const ash_map_t* map, const float* origins, const float* directions, int64_t n,
               float grid2cell, float cell_size) {
    if (check_batch(map, origins, n)) return 1;
    if (map->key_dim != 3) {
        ASH_FAIL("hashmap is not a GPU hashmap of type <int, 3>, ray sample not supported");
    }
    if (!(grid2cell > 0.f)) ASH_FAIL("grid2cell_multiplier must be positive");
    if (!(cell_size > 0.f) || !(cell_size < INFINITY)) ASH_FAIL("cell_size must be positive and finite");
    if (n > 0 && directions == nullptr) ASH_FAIL("null ray directions");
    return 0;
}

// The value of the lowest bit set in |x| (zero for zero, infinity and NaN).
float last_place(float x) {
    int e = 0;
    if (!std::isfinite(x) || x == 0.f) return 0.f;
    const auto digits = static_cast<uint32_t>(std::ldexp(std::frexp(std::fabs(x), &e), 24));
    return std::ldexp(static_cast<float>(digits & (0u - digits)), e - 24);
}

int near_far(ash_map_t* map, uint8_t* bytes, int lo, int hi, int mark, const float* origins, const float* directions, const RayUnits& units,
             const float* bbox_min, const float* bbox_max, int64_t n, float t_min, float t_max,
             float grid2cell, float* nears, float* fars, hipStream_t s) {
    if (check_rays(map, origins, directions, n, grid2cell, units.cell)) return 1;
    if (n == 0) return 0;
    if (bbox_min == nullptr || bbox_max == nullptr || nears == nullptr || fars == nullptr) {
        ASH_FAIL("null pointer in ray_find_near_far");
    }
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    if (settle_table(map, s)) return 1;
    // every step must advance t (else the march never ends), and their number
    // must stay finite
    const float half_block = static_cast<float>(grid2cell * 0.5);
    if (t_min < t_max) {
        if (!(t_max + half_block > t_max) ||
            !((static_cast<double>(t_max) - t_min) / half_block < 1e8)) {
            ASH_FAIL("ray_find_near_far: the step is too small for this range");
        }
    }
    Volume volume;
    if (make_volume(map, bytes, lo, hi, mark, volume, s)) return 1;
    StepChain chain;
    float t = t_min;
    for (int k = 0; k < kChain; ++k) {
        chain.t[k] = t;
        t += half_block;
    }
    const float per_place = 16777216.f;   // 2^24
    const float unit = last_place(half_block), start = t_min == 0.f ? unit : last_place(t_min);
    const Exact exact = {unit * per_place,
                         t_min >= 0.f && t_max + half_block <= (start < unit ? start : unit) * per_place};
    const bool pairs = volume.at != nullptr && t_min >= 0.f && t_max <= exact.near_below &&
                       (exact.steps || t >= t_max);
    if (pairs) {
        RaySteps steps = {0, 1.f / half_block};
        if (exact.steps && t_min < t_max) {
            // (a double holds all of these)
            auto below = [&](int64_t k) { return t_min + static_cast<double>(k) * half_block < t_max; };
            auto most = static_cast<int64_t>((static_cast<double>(t_max) - t_min) / half_block);
            while (most > 0 && !below(most - 1)) --most;
            while (below(most)) ++most;
            steps.most = static_cast<int>(most);
        } else {
            while (steps.most < kChain && chain.t[steps.most] < t_max) ++steps.most;
        }
        const int64_t rays = 2 * (kBlock / 64);   // per workgroup
        auto kernel = exact.steps ? ray_near_far_pairs_kernel<true> : ray_near_far_pairs_kernel<false>;
        kernel<<<static_cast<unsigned>((n + rays - 1) / rays), kBlock, 0, s>>>(
                map->d, volume, origins, directions, units, bbox_min, bbox_max, n, t_min, t_max, grid2cell,
                static_cast<float>(1.0 / grid2cell), nears, fars, steps, chain);
    } else {
        const int64_t rays = kBlock / 64;
        auto kernel = volume.at != nullptr ? ray_near_far_kernel<true> : ray_near_far_kernel<false>;
        kernel<<<static_cast<unsigned>((n + rays - 1) / rays), kBlock, 0, s>>>(
                map->d, volume, origins, directions, units, bbox_min, bbox_max, n, t_min, t_max, grid2cell,
                nears, fars, exact, chain);
    }
    ASH_LAUNCH_CHECK();
    return 0;
}

}  // namespace
}  // namespace ash

using namespace ash;

extern "C" {

int ash_ray_find_near_far(ash_map_t* map, const float* ray_origins,
                          const float* ray_directions, const float* bbox_min,
                          const float* bbox_max, int64_t n, float t_min,
                          float t_max, float t_step, float grid2cell_multiplier,
                          float* ray_nears, float* ray_fars, void* stream) {
    (void)t_step;  // unused by the reference as well (ash/src/sampler.cu:21)
    return near_far(map, nullptr, 0, 0, 0, ray_origins, ray_directions, kCellUnits, bbox_min, bbox_max, n, t_min,
                    t_max, grid2cell_multiplier, ray_nears, ray_fars,
                    static_cast<hipStream_t>(stream));
}

int64_t ash_ray_volume_bytes(int lo, int hi, int64_t n, int sampling) {
    return n < (sampling ? kVolumeRaysSampling : kVolumeRaysNearFar) ? 0 : volume_scratch(lo, hi);
}

int64_t ash_map_ray_volume_bytes(const ash_map_t* map, int lo, int hi, int64_t n, int64_t samples) {
    if (map == nullptr) return 0;
    const int64_t bytes = ash_ray_volume_bytes(lo, hi, n, samples != 0);
    const bool pays = samples == 0 ? n >= kKeptRaysNearFar : n >= kKeptRaysSampling && samples >= kKeptSamples;
    if (bytes > 0 || !pays || map->capacity > n * kKeptLogPerRay) return bytes;
    return volume_scratch(lo, hi);
}

int ash_ray_volume_kept(const ash_map_t* map, void* stream) {
    if (map == nullptr) return 0;
    DeviceGuard guard;
    // (the default stream of a device is known by the device alone)
    return guard.enter(map->device) == hipSuccess && !is_capturing(static_cast<hipStream_t>(stream)) ? 1 : 0;
}

int ash_ray_find_near_far_marked(ash_map_t* map, uint8_t* volume, int volume_lo, int volume_hi,
                                 int volume_mark, const float* ray_origins,
                                 const float* ray_directions, const float* origin, float cell_size,
                                 const float* bbox_min, const float* bbox_max, int64_t n, float t_min,
                                 float t_max, float grid2cell_multiplier, float* ray_nears,
                                 float* ray_fars, void* stream) {
    return near_far(map, volume, volume_lo, volume_hi, volume_mark, ray_origins, ray_directions,
                    {origin, 1.0f / cell_size, cell_size}, bbox_min, bbox_max, n, t_min, t_max,
                    grid2cell_multiplier, ray_nears, ray_fars, static_cast<hipStream_t>(stream));
}

int ash_ray_find_near_far_world(ash_map_t* map, uint8_t* volume, int volume_lo, int volume_hi,
                                const float* ray_origins,
                                const float* ray_directions, const float* origin, float cell_size,
                                const float* bbox_min, const float* bbox_max, int64_t n, float t_min,
                                float t_max, float grid2cell_multiplier, float* ray_nears,
                                float* ray_fars, void* stream) {
    return ash_ray_find_near_far_marked(map, volume, volume_lo, volume_hi, 0, ray_origins, ray_directions,
                                        origin, cell_size, bbox_min, bbox_max, n, t_min, t_max,
                                        grid2cell_multiplier, ray_nears, ray_fars, stream);
}

int ash_ray_sample(ash_map_t* map, const float* ray_origins,
                   const float* ray_directions, const float* ray_nears,
                   const float* ray_fars, int64_t n, int64_t max_samples_per_ray,
                   float grid2cell_multiplier, int64_t* counts,
                   const int64_t* prefix, int64_t* ray_indices, float* t_nears,
                   float* t_fars, void* stream) {
    if (check_rays(map, ray_origins, ray_directions, n, grid2cell_multiplier, 1.f)) return 1;
    if (max_samples_per_ray < 1) ASH_FAIL("max_samples_per_ray must be positive");
    if (n == 0) return 0;
    if (ray_nears == nullptr || ray_fars == nullptr) ASH_FAIL("null pointer in ray_sample");
    const bool assign = prefix != nullptr && ray_indices != nullptr &&
                        t_nears != nullptr && t_fars != nullptr;
    if ((counts != nullptr) == assign) {
        ASH_FAIL("ray_sample: pass either counts (allocation pass) or prefix and "
                 "the three outputs (assignment pass)");
    }
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (settle_table(map, s)) return 1;
    return launch_march(map, {}, {ray_origins, ray_directions, kCellUnits, ray_nears, ray_fars, 0.f, 0.f, n,
                              static_cast<float>(max_samples_per_ray), grid2cell_multiplier},
                        counts, prefix, ray_indices, t_nears, t_fars, nullptr, 0, nullptr, s);
}

int ash_ray_sample_staged(ash_map_t* map, const float* ray_origins,
                          const float* ray_directions, const float* ray_nears,
                          const float* ray_fars, int64_t n, int64_t max_samples_per_ray,
                          float grid2cell_multiplier, int64_t* counts, float* stage,
                          int64_t stride, void* stream) {
    if (check_rays(map, ray_origins, ray_directions, n, grid2cell_multiplier, 1.f)) return 1;
    if (max_samples_per_ray < 1) ASH_FAIL("max_samples_per_ray must be positive");
    if (stride < 1) ASH_FAIL("ray_sample_staged: stride must be positive");
    if (n == 0) return 0;
    if (ray_nears == nullptr || ray_fars == nullptr || counts == nullptr || stage == nullptr) {
        ASH_FAIL("null pointer in ray_sample_staged");
    }
    if (reinterpret_cast<uintptr_t>(stage) % 8 != 0) ASH_FAIL("ray_sample_staged: stage must be 8-byte aligned");
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (settle_table(map, s)) return 1;
    return launch_march(map, {}, {ray_origins, ray_directions, kCellUnits, ray_nears, ray_fars, 0.f, 0.f, n,
                              static_cast<float>(max_samples_per_ray), grid2cell_multiplier},
                        counts, nullptr, nullptr, nullptr, nullptr, stage, stride, nullptr, s);
}

int ash_ray_sample_compact(const int64_t* counts, const int64_t* prefix, const float* stage,
                           int64_t stride, int64_t n, int64_t* ray_indices, float* t_nears,
                           float* t_fars, void* stream) {
    if (n < 0 || stride < 1) ASH_FAIL("ray_sample_compact: bad sizes");
    if (n == 0) return 0;
    if (counts == nullptr || prefix == nullptr || stage == nullptr || ray_indices == nullptr ||
        t_nears == nullptr || t_fars == nullptr) {
        ASH_FAIL("null pointer in ray_sample_compact");
    }
    if (n > ((int64_t{1} << 32) - kBlock) / stride) ASH_FAIL("ray_sample_compact: too many slots");
    ray_compact_kernel<<<static_cast<unsigned>((n * stride + kBlock - 1) / kBlock), kBlock, 0,
                         static_cast<hipStream_t>(stream)>>>(
            counts, prefix, reinterpret_cast<const float2*>(stage), stride, n, ray_indices,
            t_nears, t_fars);
    ASH_LAUNCH_CHECK();
    return 0;
}

int64_t ash_ray_sample_groups(int64_t n) { return n > 0 ? static_cast<int64_t>(march_groups(n)) : 0; }

int ash_ray_sample_march_marked(ash_map_t* map, uint8_t* scratch, int volume_lo, int volume_hi,
                                int volume_mark, const float* ray_origins,
                                const float* ray_directions, const float* origin, float cell_size,
                                const float* ray_nears, const float* ray_fars, float near_for_all,
                                float far_for_all, int64_t n, int64_t max_samples_per_ray,
                                float grid2cell_multiplier, int64_t* counts, int64_t* groups,
                                float* stage, int64_t stride, int64_t out[2], void* stream) {
    if (check_rays(map, ray_origins, ray_directions, n, grid2cell_multiplier, cell_size)) return 1;
    if (max_samples_per_ray < 1) ASH_FAIL("max_samples_per_ray must be positive");
    if (stride < 1) ASH_FAIL("ray_sample_march: stride must be positive");
    if (out == nullptr) ASH_FAIL("null output pointer");
    out[0] = out[1] = 0;
    if (n == 0) return 0;
    if (counts == nullptr || groups == nullptr || stage == nullptr) {
        ASH_FAIL("null pointer in ray_sample_march");
    }
    if (reinterpret_cast<uintptr_t>(stage) % 8 != 0) ASH_FAIL("ray_sample_march: stage must be 8-byte aligned");
    if (n > (int64_t{1} << 32)) ASH_FAIL("ray_sample_march: too many rays");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (is_capturing(s)) {
        ASH_FAIL("the number of samples cannot be read while the stream is being captured");
    }
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    if (settle_table(map, s)) return 1;
    Answer answer;
    if (answer.take()) return 1;
    Volume volume;
    if (make_volume(map, scratch, volume_lo, volume_hi, volume_mark, volume, s)) return 1;
    auto* g = reinterpret_cast<GroupSamples*>(groups);
    if (launch_march(map, volume, {ray_origins, ray_directions, {origin, 1.0f / cell_size, cell_size}, ray_nears,
                           ray_fars, near_for_all, far_for_all, n,
                           static_cast<float>(max_samples_per_ray), grid2cell_multiplier},
                     counts, nullptr, nullptr, nullptr, nullptr, stage, stride, g, s)) {
        return 1;
    }
    ray_scan_kernel<<<1, kScanThreads, 0, s>>>(g, static_cast<int>(march_groups(n)), answer.words, answer.stamp);
    ASH_LAUNCH_CHECK();
    if (answer.wait(s, 4)) return 1;
    for (int w = 0; w < 2; ++w) out[w] = answer.pair(2 * w);
    return 0;
}

int ash_ray_sample_march(ash_map_t* map, uint8_t* volume, int volume_lo, int volume_hi,
                         const float* ray_origins, const float* ray_directions,
                         const float* origin, float cell_size, const float* ray_nears,
                         const float* ray_fars, float near_for_all, float far_for_all, int64_t n,
                         int64_t max_samples_per_ray, float grid2cell_multiplier, int64_t* counts,
                         int64_t* groups, float* stage, int64_t stride, int64_t out[2],
                         void* stream) {
    return ash_ray_sample_march_marked(map, volume, volume_lo, volume_hi, 0, ray_origins, ray_directions,
                                       origin, cell_size, ray_nears, ray_fars, near_for_all, far_for_all,
                                       n, max_samples_per_ray, grid2cell_multiplier, counts, groups,
                                       stage, stride, out, stream);
}

int ash_ray_sample_place(const int64_t* counts, const int64_t* groups, const float* stage,
                         int64_t stride, int64_t n, float cell_size, int64_t* ray_indices,
                         float* t_nears, float* t_fars, int64_t* prefix, void* stream) {
    if (n < 0 || stride < 1) ASH_FAIL("ray_sample_place: bad sizes");
    if (n == 0) return 0;
    if (counts == nullptr || groups == nullptr || stage == nullptr || prefix == nullptr) {
        ASH_FAIL("null pointer in ray_sample_place");
    }
    PointerGuard guard;
    ASH_HIP(guard.enter_for(counts));
    ray_place_kernel<<<march_groups(n), kBlock, 0, static_cast<hipStream_t>(stream)>>>(
            counts, reinterpret_cast<const GroupSamples*>(groups),
            reinterpret_cast<const float2*>(stage), stride, n, kBlock / lanes_per_ray(n), cell_size,
            ray_indices, t_nears, t_fars, prefix);
    ASH_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
