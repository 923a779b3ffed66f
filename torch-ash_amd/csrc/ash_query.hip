// Trilinear query kernels of libash_hip.so (gfx950): forward, backward and
// double backward of the sparse-dense grid interpolation
//   y[i,:] = sum_c w_c(offset_i) * embeddings[g_c, cell_c, :]
// with the reference's addressing (ash/src/grid.cu:68-132): the 8 corner rows
// of query i are found through three neighbour tables,
//   nbn = lut_cell_nb2grid_nb[cell_i][c]     which neighbour block (0..7)
//   g_c = lut_grid_nb2grid_idx[grid_i][nbn]  its block index, -1 if missing
//   cell_c = lut_cell_nb2cell_idx[cell_i][c] the cell inside that block
// and a query with any missing neighbour block yields zeros.
//
// Structure.  A workgroup of 256 threads takes tiles of 256 queries.
//   Phase 1 (one thread per query) reads the query's indices, offsets and mask
//   with coalesced loads, walks the neighbour tables (the two per-cell tables
//   are staged once per workgroup in LDS as uint16/uint8) and leaves the 8 row
//   numbers g_c * M + cell_c and the 3 offsets of every query in LDS.
//   Phase 2 re-maps the threads so that LPQ lanes share one query and each lane
//   owns VEC consecutive channels: one request of a wavefront then covers whole
//   embedding rows (E = 16 fp32: 4 lanes x 16 B = one 64-byte row, 16 rows per
//   instruction, 1 KiB of contiguous output), and the per-query address work is
//   not repeated per channel.  When one lane covers the row (LPQ = 1) both
//   phases run in registers without the LDS round trip.
// Workgroups are persistent and walk the tiles of "their" XCD (workgroup id
// mod 8), so neighbouring queries meet in one L2.  Gradients for the embeddings
// are accumulated with hardware floating-point atomics; consecutive queries of
// a wavefront that hit the same row are summed in registers first and issue
// one atomic per run (ray-ordered samples produce long runs).
#include "ash_query.h"

#include <type_traits>

#include <cmath>
#include <cstdlib>

namespace ash {
namespace {

// Wavefronts per SIMD, which is workgroups per CU.  Forward kernels are held to
// the 64 registers of eight, but for the widest rows (64 - 70 registers, seven),
// which would spill; the backward ones are bound by their registers (both
// gradients: 51 - 71, seven; in double precision 88 - 112, four) or by LDS.  A
// persistent grid is as many workgroups as are resident: the eighth of a CU where
// seven fit started when the others were done.  Backward of 1 - 1.5 M ray samples,
// rows of sixteen 215 -> 178 us, eight 138 -> 120, five 220 -> 206; forward of
// 2^22, rows of four, 132 -> 126.  One gradient in double precision takes 50 - 87
// registers, five to eight workgroups, and is launched with five: with as many as
// each instance has room for (the occupancy query) 1 M and 3 M ray samples took
// 0.93 - 1.08 of the time, 1.00 on average over rows of 1 to 16.
constexpr int kWavesFull = 8;
constexpr int kWavesWide = 7;
constexpr int kWavesBoth = 6;   // positions' gradient and both orders' of the rows: 60 - 78 registers
constexpr int kWavesBackward = 3;
constexpr int forward_waves(int vec, int lpq) {
    return vec > 4 || (vec == 4 && lpq > 2) ? kWavesWide : kWavesFull;
}
template <typename T>
constexpr int backward_waves(int out) {
    if (sizeof(T) == 8) return (out & 3) == 3 ? 4 : 5;
    return out == 7 ? kWavesBoth : out == 3 ? kWavesWide : kWavesFull;
}

// Runs phase 1 for the tile and hands every thread the rows / offsets of the
// query it serves in pass `p` of phase 2.
template <int LPQ, bool LDS>
struct TileStage {
    static constexpr int kPasses = LPQ;

    static __device__ __forceinline__ void fill(const QDev& a,
                                                const CellLut& lut,
                                                int64_t tile, Tile* s,
                                                uint32_t (&row)[8],
                                                float (&o)[3]) {
        fill_from(a, lut, load_inputs(a, tile * kBlock + threadIdx.x), s, row, o);
    }

    // `in`: what the calling thread's query of the tile brings (read from the
    // operand arrays, or worked out from a position by the fused front end)
    static __device__ __forceinline__ void fill_from(const QDev& a,
                                                     const CellLut& lut,
                                                     const QueryInputs& in, Tile* s,
                                                     uint32_t (&row)[8],
                                                     float (&o)[3]) {
        resolve_rows<LDS>(a, lut, in, row, o);
        if constexpr (LPQ > 1) {
            __syncthreads();  // previous tile fully consumed
#pragma unroll
            for (int c = 0; c < 8; ++c) s->row[c][threadIdx.x] = row[c];
#pragma unroll
            for (int d = 0; d < 3; ++d) s->off[d][threadIdx.x] = o[d];
            __syncthreads();
        }
    }

    static __device__ __forceinline__ int64_t fetch(int64_t tile, int p,
                                                    const Tile* s,
                                                    uint32_t (&row)[8],
                                                    float (&o)[3]) {
        if constexpr (LPQ > 1) {
            // a wavefront serves the 64 consecutive queries it resolved itself,
            // 64 / LPQ of them per pass
            const int qi = (threadIdx.x & ~63) + p * (64 / LPQ) + (threadIdx.x & 63) / LPQ;
#pragma unroll
            for (int c = 0; c < 8; ++c) row[c] = s->row[c][qi];
#pragma unroll
            for (int d = 0; d < 3; ++d) o[d] = s->off[d][qi];
            return tile * kBlock + qi;
        } else {
            return tile * kBlock + threadIdx.x;
        }
    }
};

template <typename T, int VEC>
struct VecOf;
template <>
struct VecOf<float, 4> {
    using type = float4;
};
template <>
struct VecOf<float, 1> {
    using type = float;
};
template <>
struct VecOf<float, 2> {
    using type = FloatRow<2>;
};
template <>
struct VecOf<float, 3> {
    using type = FloatRow<3>;
};
template <>
struct VecOf<float, 5> {
    using type = FloatRow<5>;
};
template <>
struct VecOf<double, 1> {
    using type = double;
};

// ------------------------------------------------------------- forward
// Phase 2 of the forward pass for the query the calling thread serves in pass
// p of the tile: gather of the eight corner rows, weighted sum, one store.
template <typename T, int VEC, int LPQ>
__device__ __forceinline__ void forward_rows(const QDev& a, const T* __restrict__ emb,
                                             T* __restrict__ out, int64_t q,
                                             const uint32_t (&row)[8], const float (&o)[3],
                                             int ch0, bool chv) {
    using V = typename VecOf<T, VEC>::type;
    const bool valid = row[0] != kNoRow;
    alignas(16) T acc[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[v] = T(0);
    if (valid && chv) {
        V e[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            e[c] = *reinterpret_cast<const V*>(
                    emb + static_cast<int64_t>(row[c]) * a.E + ch0);
        }
        AxisTerms<T> t;
        axis_terms<T, false>(o, a.smooth, t);
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const T w = corner_weight<T>(t, c);
            const T* ev = reinterpret_cast<const T*>(&e[c]);
#pragma unroll
            for (int v = 0; v < VEC; ++v) acc[v] += w * ev[v];
        }
    }
    if (q < a.N && chv) {
        if constexpr (sizeof(V) == 16) {
            typedef float v4f __attribute__((ext_vector_type(4)));
            const v4f r4 = {static_cast<float>(acc[0]), static_cast<float>(acc[VEC > 1 ? 1 : 0]),
                            static_cast<float>(acc[VEC > 2 ? 2 : 0]), static_cast<float>(acc[VEC > 3 ? 3 : 0])};
            __builtin_nontemporal_store(r4, reinterpret_cast<v4f*>(out + q * a.E + ch0));
        } else {
#pragma unroll
            for (int v = 0; v < VEC; ++v) {
                __builtin_nontemporal_store(acc[v], out + q * a.E + ch0 + v);
            }
        }
    }
}

template <typename T, int VEC, int LPQ, bool LDS>
__global__ __launch_bounds__(kBlock, forward_waves(VEC, LPQ)) void
query_forward_kernel(
        QDev a, T* __restrict__ out) {
    extern __shared__ __align__(16) unsigned char smem[];
    Tile* tile_s = reinterpret_cast<Tile*>(smem);
    const CellLut lut =
            stage_cell_lut<LDS>(a, smem + (LPQ > 1 ? sizeof(Tile) : 0));
    using Stage = TileStage<LPQ, LDS>;
    const int ch0 = (threadIdx.x % LPQ) * VEC;
    const bool chv = ch0 < a.E;
    const T* __restrict__ emb = static_cast<const T*>(a.emb);
    const int64_t ntiles = (a.N + kBlock - 1) / kBlock;
    TileWalk walk(ntiles);
    for (int64_t tile = walk.next; tile < walk.end; tile += walk.step) {
        uint32_t row[8];
        float o[3];
        Stage::fill(a, lut, tile, tile_s, row, o);
#pragma unroll 1
        for (int p = 0; p < Stage::kPasses; ++p) {
            const int64_t q = Stage::fetch(tile, p, tile_s, row, o);
            forward_rows<T, VEC, LPQ>(a, emb, out, q, row, o, ch0, chv);
        }
    }
}

// ------------------------------------------------ forward from positions
// The module-level forward (ash/grid.py:201-238: `query`, then the
// interpolation) in one kernel: the front end of ash_grid_query (position ->
// block / cell / fractional part -> look-up of the block, ash_probe.h) stands
// where the forward kernel reads a query's operands, so the four intermediate
// arrays are neither written nor read back on the way to the result -- they are
// written (once) only for a caller that needs them afterwards: the mask always
// (the module returns it), block index, cell index and offsets when a backward
// pass will want them (AUX).
struct FrontDev {
    MapDev m;
    const float* x;      // float32[N, 3]; cell units = (x - origin) * inv_cell
    const float* origin; // float32[3] on the device, or nullptr for none
    float inv_cell;      // 1 / cell size, rounded to fp32 once
    float g;             // cells per block edge
    int gdim;
    uint8_t* mask_out;   // [N]
    int64_t* gidx_out;   // [N]    (AUX)
    int64_t* cidx_out;   // [N]    (AUX)
    float* off_out;      // [N, 3] (AUX)
};

__device__ __forceinline__ void load_position(const QDev& a, const FrontDev& f, int64_t q,
                                              float (&x)[3]) {
#pragma unroll
    for (int d = 0; d < 3; ++d) x[d] = q < a.N ? __builtin_nontemporal_load(f.x + q * 3 + d) : 0.f;
}

template <bool AUX>
__device__ __forceinline__ QueryInputs front_inputs(const QDev& a, const FrontDev& f, int64_t q,
                                                    const float (&x)[3]) {
    const bool active = q < a.N;
    QueryInputs in;
    int32_t k[3];
    int32_t cell = 0, stride = 1;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        int32_t c;
        float xv = x[d];
        // world -> cell units the way torch evaluates `(x - origin) / cell_size`
        // on the device: a subtraction, then a multiplication by the fp32
        // reciprocal of the size (both exact no-ops for origin 0 and size 1)
        xv = __fmul_rn(__fsub_rn(xv, f.origin != nullptr ? f.origin[d] : 0.f), f.inv_cell);
        split_axis(xv, f.g, k[d], c, in.o[d]);
        cell += c * stride;
        stride *= f.gdim;
    }
    int32_t res = 0;
    const bool found = find_block_by_runs(f.m, k, active, res);
    in.gi = found ? res : 0;
    in.ci = cell;
    in.m = (active && found) ? 1 : 0;
    if (active) {
        __builtin_nontemporal_store(in.m, f.mask_out + q);
        if constexpr (AUX) {
            __builtin_nontemporal_store(static_cast<int64_t>(in.gi), f.gidx_out + q);
            __builtin_nontemporal_store(static_cast<int64_t>(cell), f.cidx_out + q);
#pragma unroll
            for (int d = 0; d < 3; ++d) __builtin_nontemporal_store(in.o[d], f.off_out + q * 3 + d);
        }
    }
    return in;
}

template <typename T, int VEC, int LPQ, bool LDS, bool AUX>
__global__ __launch_bounds__(kBlock, forward_waves(VEC, LPQ)) void
grid_forward_kernel(QDev a, FrontDev f, T* __restrict__ out) {
    extern __shared__ __align__(16) unsigned char smem[];
    Tile* tile_s = reinterpret_cast<Tile*>(smem);
    const CellLut lut =
            stage_cell_lut<LDS>(a, smem + (LPQ > 1 ? sizeof(Tile) : 0));
    using Stage = TileStage<LPQ, LDS>;
    const int ch0 = (threadIdx.x % LPQ) * VEC;
    const bool chv = ch0 < a.E;
    const T* __restrict__ emb = static_cast<const T*>(a.emb);
    const int64_t ntiles = (a.N + kBlock - 1) / kBlock;
    TileWalk walk(ntiles);
    // (the positions come from memory, the longest of a tile's trips: a tile
    // ahead.  Rows of 8: 42 -> 40 us, blocks of 16^3: 43 -> 40, others 0 - 3 %;
    // the other kernels lose as much as they gain by it)
    const auto first_of = [&](int64_t tile) {
        return tile < walk.end ? tile * kBlock + threadIdx.x : a.N;
    };
    float ahead[3];
    load_position(a, f, first_of(walk.next), ahead);
    for (int64_t tile = walk.next; tile < walk.end; tile += walk.step) {
        uint32_t row[8];
        float o[3];
        const float x[3] = {ahead[0], ahead[1], ahead[2]};
        load_position(a, f, first_of(tile + walk.step), ahead);
        Stage::fill_from(a, lut, front_inputs<AUX>(a, f, tile * kBlock + threadIdx.x, x), tile_s,
                         row, o);
#pragma unroll 1
        for (int p = 0; p < Stage::kPasses; ++p) {
            const int64_t q = Stage::fetch(tile, p, tile_s, row, o);
            forward_rows<T, VEC, LPQ>(a, emb, out, q, row, o, ch0, chv);
        }
    }
}

// ------------------------------------------------- run merge for atomics
// Runs of consecutive queries of a wavefront that lie in the same cell.  Two
// queries meet in the same row at a corner only when they lie in the same
// cell, and then at every corner, so the runs are found once per pass, from
// the row of the cell itself, and the sums over them are taken corner by
// corner: one lane exchange per step and corner.  Query groups are LPQ lanes
// wide (one lane per channel); a lane talks to the lanes of its own channel.
template <int LPQ>
struct GroupRuns {
    static constexpr int kGroups = 64 / LPQ;
    static constexpr int kSteps = kGroups > 32 ? 6 : kGroups > 16 ? 5 : kGroups > 8 ? 4
                                  : kGroups > 4 ? 3 : kGroups > 2 ? 2 : 1;
    bool any;            // some group continues the run of the group before it (the same for all lanes)
    bool take[kSteps];   // step k of the segmented sum adds what lies 2^k groups below
    bool tail;           // the last group of its run: holds the total afterwards
};

// `on`: the lane has a query and a channel.  Every lane of the wavefront must
// take part.
template <int LPQ>
__device__ __forceinline__ GroupRuns<LPQ> find_group_runs(uint32_t cell_row, bool on, int lane) {
    using R = GroupRuns<LPQ>;
    R r;
    const int grp = lane / LPQ;
    // lanes that are off get a row number no neighbour shares
    const uint32_t id = on ? cell_row : (kNoRow - static_cast<uint32_t>(grp & 1));
    const uint32_t prev = __shfl_up(id, LPQ);
    const uint32_t next = __shfl_down(id, LPQ);
    const bool head = (grp == 0) || (prev != id) || !on;
    r.tail = (grp == R::kGroups - 1) || (next != id);
    r.any = __ballot(!head) != 0;
    int f = head ? 1 : 0;
#pragma unroll
    for (int k = 0; k < R::kSteps; ++k) {
        const int d = 1 << k;
        const int fu = __shfl_up(f, d * LPQ);
        r.take[k] = grp >= d && !f;
        if (r.take[k]) f |= fu;
    }
    return r;
}

// Adds v to grad_emb[row, ch] for the lanes that are `on`; with `runs` the
// last group of every run adds the run's sum (runs.any false: every lane for
// itself).  Every lane of the wavefront must take part.
template <typename T, int LPQ>
__device__ __forceinline__ void accumulate_row(T* __restrict__ grad_emb,
                                               uint32_t row, int E, int ch,
                                               bool on, T v, const GroupRuns<LPQ>& runs) {
    bool last = true;
    if (runs.any) {   // (the same for all lanes)
#pragma unroll
        for (int k = 0; k < GroupRuns<LPQ>::kSteps; ++k) {
            const T vu = __shfl_up(v, (1 << k) * LPQ);
            if (runs.take[k]) v += vu;
        }
        last = runs.tail;
    }
    if (on && last) {
        unsafeAtomicAdd(grad_emb + static_cast<int64_t>(row) * E + ch, v);
    }
}

// --------------------------------------------------- backward (first order)
// grad_embeddings[row_c, k] += w_c * z[i,k];
// grad_offsets[i,:] = sum_c (emb[row_c,:] . z[i,:]) * grad w_c
// (ash/src/grid.cu:177-255).  One lane per channel.
// OUT: bit 0 = produce grad_embeddings, bit 1 = produce grad_offsets; bit 2 (with
// bit 0) = and add to grad_embeddings what the backward of the backward does for
// gg_off and z2 (below): the two contributions of a query go to the same eight
// rows, and the requests for these are what either kernel is bound by (positions'
// gradient and rows of sixteen, 131 k ray samples: 52 + 39 -> 62 us, 500 k 122 + 99 ->
// 136; 2^22, rows of four, in the kernel for these: 187 + 184 -> 254).  Rows of 1 to 8
// and 12 floats as a rule go by the kernels for whole rows (rows_by_lane).
template <typename T, int LPQ, bool LDS, int OUT>
__global__ __launch_bounds__(kBlock, kWavesBackward) void
query_backward_forward_kernel(
        QDev a, const T* __restrict__ z, T* __restrict__ grad_emb,
        T* __restrict__ grad_off, const T* __restrict__ gg_off, const T* __restrict__ z2) {
    extern __shared__ __align__(16) unsigned char smem[];
    Tile* tile_s = reinterpret_cast<Tile*>(smem);
    const CellLut lut =
            stage_cell_lut<LDS>(a, smem + (LPQ > 1 ? sizeof(Tile) : 0));
    using Stage = TileStage<LPQ, LDS>;
    const int lane = threadIdx.x & 63;
    const int ch = threadIdx.x % LPQ;
    const bool chv = ch < a.E;
    const T* __restrict__ emb = static_cast<const T*>(a.emb);
    constexpr bool want_emb = (OUT & 1) != 0;
    constexpr bool want_off = (OUT & 2) != 0;
    constexpr bool second = (OUT & 4) != 0;
    const int64_t ntiles = (a.N + kBlock - 1) / kBlock;
    TileWalk walk(ntiles);
    for (int64_t tile = walk.next; tile < walk.end; tile += walk.step) {
        uint32_t row[8];
        float o[3];
        Stage::fill(a, lut, tile, tile_s, row, o);
#pragma unroll 1
        for (int p = 0; p < Stage::kPasses; ++p) {
            const int64_t q = Stage::fetch(tile, p, tile_s, row, o);
            const bool valid = row[0] != kNoRow;
            const bool on = valid && chv;
            const T zk = on ? z[q * a.E + ch] : T(0);
            T zk2 = T(0), gg[3] = {T(0), T(0), T(0)};
            if constexpr (second) {
                if (on) zk2 = z2[q * a.E + ch];
                if (valid) {
                    gg[0] = gg_off[q * 3 + 0] * static_cast<T>(a.offset_scale);
                    gg[1] = gg_off[q * 3 + 1] * static_cast<T>(a.offset_scale);
                    gg[2] = gg_off[q * 3 + 2] * static_cast<T>(a.offset_scale);
                }
            }
            GroupRuns<LPQ> runs;
            runs.any = false;
            if (want_emb && a.merge) runs = find_group_runs<LPQ>(row[0], on, lane);
            T e[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                e[c] = (on && want_off)
                               ? emb[static_cast<int64_t>(row[c]) * a.E + ch]
                               : T(0);
            }
            AxisTerms<T> t;
            axis_terms<T, true>(o, a.smooth, t);
            SlopeTerms<T> slope;
            if constexpr (second) slope_terms<T>(t, gg, slope);
            T go[3] = {T(0), T(0), T(0)};
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                if constexpr (want_emb) {
                    const T w = corner_weight<T>(t, c);
                    T v = w * zk;
                    if constexpr (second) v += corner_slope<T>(t, slope, c) * zk2;
                    accumulate_row<T, LPQ>(grad_emb, row[c], a.E, ch, on, v, runs);
                }
                if constexpr (want_off) {
                    T gw[3];
                    corner_weight_grad<T>(t, c, gw);
                    T dot = e[c] * zk;
#pragma unroll
                    for (int s = 1; s < LPQ; s <<= 1) dot += __shfl_xor(dot, s);
                    go[0] += dot * gw[0];
                    go[1] += dot * gw[1];
                    go[2] += dot * gw[2];
                }
            }
            if (want_off && q < a.N && ch == 0) {
                const T scale = static_cast<T>(a.offset_scale);
                grad_off[q * 3 + 0] = valid ? go[0] * scale : T(0);
                grad_off[q * 3 + 1] = valid ? go[1] * scale : T(0);
                grad_off[q * 3 + 2] = valid ? go[2] * scale : T(0);
            }
        }
    }
}

// -------------------------------------------------- backward of backward
// d_c = grad w_c . gg_off[i];  grad_embeddings[row_c,k] += d_c * z[i,k];
// grad_z[i,k] = sum_c d_c * emb[row_c,k]   (ash/src/grid.cu:309-387).
// OUT: bit 0 = produce grad_embeddings, bit 1 = produce grad_z.
template <typename T, int LPQ, bool LDS, int OUT>
__global__ __launch_bounds__(kBlock, kWavesBackward) void
query_backward_backward_kernel(
        QDev a, const T* __restrict__ gg_off, const T* __restrict__ z,
        T* __restrict__ grad_z, T* __restrict__ grad_emb) {
    extern __shared__ __align__(16) unsigned char smem[];
    Tile* tile_s = reinterpret_cast<Tile*>(smem);
    const CellLut lut =
            stage_cell_lut<LDS>(a, smem + (LPQ > 1 ? sizeof(Tile) : 0));
    using Stage = TileStage<LPQ, LDS>;
    const int lane = threadIdx.x & 63;
    const int ch = threadIdx.x % LPQ;
    const bool chv = ch < a.E;
    const T* __restrict__ emb = static_cast<const T*>(a.emb);
    constexpr bool want_emb = (OUT & 1) != 0;
    constexpr bool want_z = (OUT & 2) != 0;
    const int64_t ntiles = (a.N + kBlock - 1) / kBlock;
    TileWalk walk(ntiles);
    for (int64_t tile = walk.next; tile < walk.end; tile += walk.step) {
        uint32_t row[8];
        float o[3];
        Stage::fill(a, lut, tile, tile_s, row, o);
#pragma unroll 1
        for (int p = 0; p < Stage::kPasses; ++p) {
            const int64_t q = Stage::fetch(tile, p, tile_s, row, o);
            const bool valid = row[0] != kNoRow;
            const bool on = valid && chv;
            const T zk = on ? z[q * a.E + ch] : T(0);
            GroupRuns<LPQ> runs;
            runs.any = false;
            if (want_emb && a.merge) runs = find_group_runs<LPQ>(row[0], on, lane);
            T gg[3] = {T(0), T(0), T(0)};
            if (valid) {
                gg[0] = gg_off[q * 3 + 0] * static_cast<T>(a.offset_scale);
                gg[1] = gg_off[q * 3 + 1] * static_cast<T>(a.offset_scale);
                gg[2] = gg_off[q * 3 + 2] * static_cast<T>(a.offset_scale);
            }
            T e[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                e[c] = (on && want_z)
                               ? emb[static_cast<int64_t>(row[c]) * a.E + ch]
                               : T(0);
            }
            AxisTerms<T> t;
            axis_terms<T, true>(o, a.smooth, t);
            T gz = T(0);
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                T gw[3];
                corner_weight_grad<T>(t, c, gw);
                const T d = gw[0] * gg[0] + gw[1] * gg[1] + gw[2] * gg[2];
                if constexpr (want_emb) {
                    accumulate_row<T, LPQ>(grad_emb, row[c], a.E, ch, on, d * zk, runs);
                }
                gz += d * e[c];
            }
            if (want_z && q < a.N && chv) {
                grad_z[q * a.E + ch] = on ? gz : T(0);
            }
        }
    }
}

// Sparse convolution forward (ash/src/grid.cu:948-1043): for every cell of the
// listed blocks, out[row] = sum over the K window taps k of
// in[row of neighbour k] * w[k], channel by channel, taps whose block is
// missing skipped.  One lane per (cell, channel): a wavefront reads whole rows
// of neighbouring cells, and the taps are accumulated in the reference's order
// with one fused multiply-add each (what nvcc makes of `sum += in * w`).
struct ConvDev {
    const void* in;
    const void* w;
    const uint8_t* masks;
    const int64_t* grid_indices;
    const int64_t* cell_indices;
    const int64_t* lut_g;     // [B, GN]
    const int64_t* lut_c2c;   // [M, K]
    const int64_t* lut_c2g;   // [M, K]
    void* out;
    int64_t n_grids, B, M, E, K, GN;
    int owns;   // the kernel writes every cell of the listed blocks (zeros where it has no result)
};

// One lane per cell with all channels of the row in registers (EC >= E, a
// power of two up to 16): consecutive lanes are consecutive cells, so a tap
// reads a contiguous run of rows, and the table entries are fetched once per
// cell instead of once per channel.  `vec4`: fp32 rows of a multiple of four
// channels on 16-byte aligned buffers are moved as float4.
template <typename T, int EC>
__global__ __launch_bounds__(kBlock) void convolution_cell_kernel(ConvDev a, int vec4) {
    const int64_t item = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (item >= a.n_grids * a.M || !a.masks[item]) return;
    const int64_t g = a.grid_indices[item / a.M];
    const int64_t c = a.cell_indices[item % a.M];
    if (g < 0 || g >= a.B || c < 0 || c >= a.M) return;
    const T* in = static_cast<const T*>(a.in);
    const T* w = static_cast<const T*>(a.w);
    const int64_t* nb_g = a.lut_g + g * a.GN;
    const int64_t* nb_c = a.lut_c2c + c * a.K;
    const int64_t* nb_n = a.lut_c2g + c * a.K;
    const int E = static_cast<int>(a.E);
    T acc[EC];
#pragma unroll
    for (int e = 0; e < EC; ++e) acc[e] = T(0);
    for (int64_t k = 0; k < a.K; ++k) {
        const int64_t gn = nb_n[k];
        if (gn < 0 || gn >= a.GN) continue;
        const int64_t gi = nb_g[gn];
        if (gi < 0 || gi >= a.B) continue;
        const int64_t ci = nb_c[k];
        if (ci < 0 || ci >= a.M) continue;
        const T* row = in + (gi * a.M + ci) * E;
        const T* wk = w + k * E;
        if constexpr (sizeof(T) == 4 && EC >= 4) {
            if (vec4) {
#pragma unroll
                for (int q = 0; q < EC / 4; ++q) {
                    if (4 * q < E) {
                        const float4 r = reinterpret_cast<const float4*>(row)[q];
                        acc[4 * q + 0] = fmaf(r.x, wk[4 * q + 0], acc[4 * q + 0]);
                        acc[4 * q + 1] = fmaf(r.y, wk[4 * q + 1], acc[4 * q + 1]);
                        acc[4 * q + 2] = fmaf(r.z, wk[4 * q + 2], acc[4 * q + 2]);
                        acc[4 * q + 3] = fmaf(r.w, wk[4 * q + 3], acc[4 * q + 3]);
                    }
                }
                continue;
            }
        }
#pragma unroll
        for (int e = 0; e < EC; ++e) {
            if (e < E) acc[e] = fma(row[e], wk[e], acc[e]);
        }
    }
    T* o = static_cast<T*>(a.out) + (g * a.M + c) * E;
    if constexpr (sizeof(T) == 4 && EC >= 4) {
        if (vec4) {
#pragma unroll
            for (int q = 0; q < EC / 4; ++q) {
                if (4 * q < E) {
                    reinterpret_cast<float4*>(o)[q] = make_float4(
                            acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
                }
            }
            return;
        }
    }
#pragma unroll
    for (int e = 0; e < EC; ++e) {
        if (e < E) o[e] = acc[e];
    }
}

// The same per-cell accumulation with one persistent workgroup per block of
// cells at a time: the block's own rows are staged in LDS (for a 3^3 window
// about four taps in five stay inside the block) and the two per-cell tables
// are kept in LDS in compact form (uint16 cell, uint8 block offset) for the
// whole launch, when they fit.  Taps, order and arithmetic are unchanged.
constexpr int kConvThreads = 512;

template <typename T, int EC>
__global__ __launch_bounds__(kConvThreads) void convolution_block_kernel(
        ConvDev a, int vec4, int lut_lds, int rows_lds) {
    extern __shared__ __align__(16) unsigned char conv_smem[];
    const int tid = threadIdx.x;
    const int E = static_cast<int>(a.E);
    const int M = static_cast<int>(a.M);
    const int K = static_cast<int>(a.K);
    T* rows = reinterpret_cast<T*>(conv_smem);
    const size_t rows_bytes =
            rows_lds ? (static_cast<size_t>(M) * E * sizeof(T) + 15) / 16 * 16 : 0;
    uint16_t* cc = reinterpret_cast<uint16_t*>(conv_smem + rows_bytes);
    uint8_t* cg = reinterpret_cast<uint8_t*>(cc + static_cast<size_t>(M) * K);
    if (lut_lds) {
        for (int t = tid; t < M * K; t += kConvThreads) {
            const int64_t ci = a.lut_c2c[t];
            const int64_t gn = a.lut_c2g[t];
            cc[t] = (ci >= 0 && ci < M) ? static_cast<uint16_t>(ci) : 0xFFFFu;
            cg[t] = (gn >= 0 && gn < a.GN) ? static_cast<uint8_t>(gn) : 0xFFu;
        }
    }
    const T* in = static_cast<const T*>(a.in);
    const T* w = static_cast<const T*>(a.w);
    for (int64_t blk = blockIdx.x; blk < a.n_grids; blk += gridDim.x) {
        const int64_t g = a.grid_indices[blk];
        const bool g_ok = g >= 0 && g < a.B;
        __syncthreads();
        if (rows_lds && g_ok) {
            const T* src = in + g * a.M * E;
            if (vec4) {
                for (int t = tid; t < M * E / 4; t += kConvThreads) {
                    reinterpret_cast<float4*>(rows)[t] = reinterpret_cast<const float4*>(src)[t];
                }
            } else {
                for (int t = tid; t < M * E; t += kConvThreads) rows[t] = src[t];
            }
        }
        __syncthreads();
        if (!g_ok) continue;
        const int64_t* nb_g = a.lut_g + g * a.GN;
        for (int c_i = tid; c_i < M; c_i += kConvThreads) {
            if (!a.masks[blk * a.M + c_i]) continue;
            const int64_t c = a.cell_indices[c_i];
            if (c < 0 || c >= a.M) continue;
            T acc[EC];
#pragma unroll
            for (int e = 0; e < EC; ++e) acc[e] = T(0);
            for (int k = 0; k < K; ++k) {
                int64_t gn, ci;
                if (lut_lds) {
                    const uint16_t ci16 = cc[c * K + k];
                    const uint8_t gn8 = cg[c * K + k];
                    if (ci16 == 0xFFFFu || gn8 == 0xFFu) continue;
                    ci = ci16;
                    gn = gn8;
                } else {
                    gn = a.lut_c2g[c * K + k];
                    ci = a.lut_c2c[c * K + k];
                    if (gn < 0 || gn >= a.GN || ci < 0 || ci >= a.M) continue;
                }
                const int64_t gi = nb_g[gn];
                if (gi < 0 || gi >= a.B) continue;
                const T* row = (rows_lds && gi == g) ? rows + ci * E
                                                     : in + (gi * a.M + ci) * E;
                const T* wk = w + static_cast<int64_t>(k) * E;
                if constexpr (sizeof(T) == 4 && EC >= 4) {
                    if (vec4) {
#pragma unroll
                        for (int q = 0; q < EC / 4; ++q) {
                            if (4 * q < E) {
                                const float4 r = reinterpret_cast<const float4*>(row)[q];
                                acc[4 * q + 0] = fmaf(r.x, wk[4 * q + 0], acc[4 * q + 0]);
                                acc[4 * q + 1] = fmaf(r.y, wk[4 * q + 1], acc[4 * q + 1]);
                                acc[4 * q + 2] = fmaf(r.z, wk[4 * q + 2], acc[4 * q + 2]);
                                acc[4 * q + 3] = fmaf(r.w, wk[4 * q + 3], acc[4 * q + 3]);
                            }
                        }
                        continue;
                    }
                }
#pragma unroll
                for (int e = 0; e < EC; ++e) {
                    if (e < E) acc[e] = fma(row[e], wk[e], acc[e]);
                }
            }
            T* o = static_cast<T*>(a.out) + (g * a.M + c) * E;
            bool stored = false;
            if constexpr (sizeof(T) == 4 && EC >= 4) {
                if (vec4) {
#pragma unroll
                    for (int q = 0; q < EC / 4; ++q) {
                        if (4 * q < E) {
                            reinterpret_cast<float4*>(o)[q] = make_float4(
                                    acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
                        }
                    }
                    stored = true;
                }
            }
            if (!stored) {
#pragma unroll
                for (int e = 0; e < EC; ++e) {
                    if (e < E) o[e] = acc[e];
                }
            }
        }
    }
}

template <typename T, int EC>
int launch_convolution_block(const ConvDev& a, int vec4, hipStream_t s) {
    const size_t rows_bytes = (static_cast<size_t>(a.M) * a.E * sizeof(T) + 15) / 16 * 16;
    const size_t lut_bytes = static_cast<size_t>(a.M) * a.K * 3;
    const int rows_lds = rows_bytes <= 64 * 1024 ? 1 : 0;
    const int lut_lds = (lut_bytes <= 48 * 1024 && a.M < 0xFFFF && a.GN < 0xFF) ? 1 : 0;
    const size_t smem = (rows_lds ? rows_bytes : 0) + (lut_lds ? lut_bytes : 0) + 16;
    auto kernel = convolution_block_kernel<T, EC>;
    ASH_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                static_cast<int>(smem)));
    unsigned g = persistent_grid(a.n_grids, smem);
    kernel<<<g, kConvThreads, smem, s>>>(a, vec4, lut_lds, rows_lds);
    ASH_LAUNCH_CHECK();
    return 0;
}

// Cube windows over cubic blocks in the layout the Python layer builds
// (cell c = x + G y + G^2 z; tap k = (dx + r) + W (dy + r) + W^2 (dz + r) with
// W = 2 r + 1; neighbour block (bx + 1) + 3 (by + 1) + 9 (bz + 1)): the block's
// cells together with their halo of r cells, (G + 2r)^3 rows of EC channels,
// are staged in LDS once per block, and every cell then reads its W^3 taps from
// there -- in table order, one fused multiply-add per tap and channel, like the
// other kernels.  Rows of missing blocks are staged as zeros: with finite
// weights adding 0 * w leaves the accumulator as it is (it starts at +0 and so
// never is -0), which is what skipping the tap does.  Every workgroup first
// checks the two per-cell tables against this layout and, should they describe
// something else, takes its blocks through the tables instead.
// EC: channels per pass; WT: window edge when it is 3, 5 or 7, else 0; NY: cells
// per lane along y (0: one lane = one cell with all EC channels).
// The second launch bound asks for four wavefronts per SIMD (two workgroups
// per CU, at most 128 registers) for all but the widest instances, which need
// more registers than that for their window.
template <typename T, int EC, int WT, int NY>
__global__ __launch_bounds__(kConvThreads, (EC >= 16 && NY >= 8) ? 2 : 4) void convolution_tile_kernel(
        ConvDev a, int G, int r, int e0, int ec, int vec, int Tz) {
    constexpr bool YB = NY > 0;   // NY cells that follow each other in y per lane
    extern __shared__ __align__(16) unsigned char conv_smem[];
    __shared__ int64_t s_nb[2][28];   // rows of 27 neighbour blocks + the block itself
    __shared__ int s_bad;
    const int tid = threadIdx.x;
    const int E = static_cast<int>(a.E);
    const int M = static_cast<int>(a.M);
    const int K = static_cast<int>(a.K);
    const int W = WT > 0 ? WT : 2 * r + 1;   // WT: window edge known at compile time
    const int Tn = G + 2 * r;
    const int T3 = Tn * Tn * Tn;
    // Tz: words from one z layer of a channel's plane to the next, Tn * Tn or
    // a little more (YB): the lanes of a wavefront read G words along x at
    // NY * Tn words from one group of lanes to the next in y and Tz in z, and
    // the host pads Tz so that the groups served together fall on different
    // LDS banks.
    const int Ts = Tz * Tn;        // words of one channel's plane
    const int zpad = Tz - Tn * Tn;
    T* tile = reinterpret_cast<T*>(conv_smem);                             // [Ts][EC]
    T* s_w = tile + static_cast<size_t>(Ts) * EC;                          // [K][EC]
    uint32_t* s_src = reinterpret_cast<uint32_t*>(s_w + static_cast<size_t>(K) * EC);  // [T3]
    uint16_t* s_inv = reinterpret_cast<uint16_t*>(s_src + T3);   // [M] position of a cell in cell_indices (YB)
    // YB keeps one plane per channel (a lane reads runs of one channel along
    // x), otherwise the channels of a row sit together.  p counts the rows of
    // the tile without the padding.
    auto plane_at = [&](int p) { return p + zpad * (p / (Tn * Tn)); };
    auto tile_at = [&](int p, int q) { return YB ? q * Ts + plane_at(p) : p * EC + q; };
    auto w_at = [&](int k, int q) { return YB ? q * K + k : k * EC + q; };
    const T* in = static_cast<const T*>(a.in);
    const T* w = static_cast<const T*>(a.w);
    T* out = static_cast<T*>(a.out);

    if (tid == 0) s_bad = 0;
    __syncthreads();
    {
        int bad = 0;
        for (int t = tid; t < M * K; t += kConvThreads) {
            const int c = t / K;
            const int k = t - c * K;
            const int x[3] = {c % G, (c / G) % G, c / (G * G)};
            const int o[3] = {k % W - r, (k / W) % W - r, k / (W * W) - r};
            int gn = 0, ci = 0, gs = 1, cs = 1;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const int t_d = x[d] + o[d];
                const int b = t_d < 0 ? -1 : (t_d >= G ? 1 : 0);
                gn += (b + 1) * gs;
                ci += (t_d - b * G) * cs;
                gs *= 3;
                cs *= G;
            }
            bad |= a.lut_c2g[t] != gn || a.lut_c2c[t] != ci;
        }
        if (bad) s_bad = 1;
        // where every row of the tile comes from and where it goes:
        // place in the tile << 17 | neighbour block << 12 | cell
        for (int p = tid; p < T3; p += kConvThreads) {
            const int tx[3] = {p % Tn - r, (p / Tn) % Tn - r, p / (Tn * Tn) - r};
            int gn = 0, ci = 0, gs = 1, cs = 1;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const int b = tx[d] < 0 ? -1 : (tx[d] >= G ? 1 : 0);
                gn += (b + 1) * gs;
                ci += (tx[d] - b * G) * cs;
                gs *= 3;
                cs *= G;
            }
            s_src[p] = (static_cast<uint32_t>(tile_at(p, 0)) << 17) | static_cast<uint32_t>((gn << 12) | ci);
        }
        for (int t = tid; t < K * EC; t += kConvThreads) {
            const int k = t / EC;
            const int q = t - k * EC;
            s_w[w_at(k, q)] = q < ec ? w[k * E + e0 + q] : T(0);
        }
        if constexpr (YB) {
            for (int c = tid; c < M; c += kConvThreads) s_inv[c] = 0xFFFFu;
        }
    }
    __syncthreads();
    if constexpr (YB) {
        for (int c_i = tid; c_i < M; c_i += kConvThreads) {
            const int64_t c = a.cell_indices[c_i];
            if (c >= 0 && c < a.M) s_inv[c] = static_cast<uint16_t>(c_i);
        }
    }
    __syncthreads();
    const bool by_table = s_bad != 0;

    // a.owns: nobody cleared the rows of the listed blocks, so cells without a
    // result get their zeros here.  The paths that visit cells through
    // cell_indices clear the whole block first, in the pass of the first
    // channels; the y-blocked path writes a zero where it skips a cell.
    auto clear_block = [&](int64_t g) {
        if (!a.owns || e0 != 0) return;
        T* rows = out + g * a.M * a.E;
        for (int64_t i = tid; i < a.M * a.E; i += kConvThreads) rows[i] = T(0);
        __syncthreads();
    };
    for (int64_t blk = blockIdx.x; by_table && blk < a.n_grids; blk += gridDim.x) {
        const int64_t g = a.grid_indices[blk];
        if (g < 0 || g >= a.B) continue;  // the same for the whole workgroup
        clear_block(g);
        {
            const int64_t* nb_g = a.lut_g + g * a.GN;
            for (int c_i = tid; c_i < M; c_i += kConvThreads) {
                if (!a.masks[blk * a.M + c_i]) continue;
                const int64_t c = a.cell_indices[c_i];
                if (c < 0 || c >= a.M) continue;
                T acc[EC];
#pragma unroll
                for (int q = 0; q < EC; ++q) acc[q] = T(0);
                for (int k = 0; k < K; ++k) {
                    const int64_t gn = a.lut_c2g[c * K + k];
                    if (gn < 0 || gn >= a.GN) continue;
                    const int64_t gi = nb_g[gn];
                    if (gi < 0 || gi >= a.B) continue;
                    const int64_t ci = a.lut_c2c[c * K + k];
                    if (ci < 0 || ci >= a.M) continue;
#pragma unroll
                    for (int q = 0; q < EC; ++q) {
                        if (q < ec) {
                            acc[q] = fma(in[(gi * a.M + ci) * E + e0 + q], s_w[w_at(k, q)], acc[q]);
                        }
                    }
                }
#pragma unroll
                for (int q = 0; q < EC; ++q) {
                    if (q < ec) out[(g * a.M + c) * E + e0 + q] = acc[q];
                }
            }
        }
    }
    if (by_table) return;

    // Blocks through the tile, software-pipelined: while a block is computed
    // from LDS, the rows of the next block's tile are already on their way
    // into registers and the row numbers of the block after that are fetched.
    // each XCD walks a contiguous eighth of the listing (TileWalk): with blocks
    // listed along a space-filling curve the halo rows are then mostly in the
    // XCD's own L2
    const TileWalk walk(a.n_grids);
    constexpr int kPre = EC >= 16 ? 2 : (EC >= 8 ? 4 : 6);   // tile rows a thread can hold
    const bool prefetch = T3 <= kPre * kConvThreads;
    auto fetch_rows = [&](int64_t b) -> int64_t {  // lanes 0..26 neighbours, 27 the block
        if (tid > 27 || b >= walk.end) return -1;
        const int64_t g = a.grid_indices[b];
        if (g < 0 || g >= a.B) return -1;
        if (tid == 27) return g;
        const int64_t row = a.lut_g[g * 27 + tid];
        return (row >= 0 && row < a.B) ? row : -1;
    };
    // src_cell: an entry of s_src, or kNoRow for a thread without a row
    constexpr uint32_t kNoRow = 0xFFFFFFFFu;
    const T* in_e0 = in + e0;
    const uint32_t block_words = static_cast<uint32_t>(M * E);   // <= 4096 * 16
    auto load_row = [&](const int64_t* nb, uint32_t src_cell, T (&v)[EC]) {
#pragma unroll
        for (int q = 0; q < EC; ++q) v[q] = T(0);
        if (src_cell == kNoRow) return;
        const int64_t row = nb[(src_cell >> 12) & 31];
        if (row < 0) return;
        // row < B < 2^31: one 32 x 32 -> 64 bit product
        const T* src = in_e0 + (static_cast<uint64_t>(static_cast<uint32_t>(row)) * block_words +
                                (src_cell & 0xFFF) * static_cast<uint32_t>(E));
        if (vec) {   // EC is a multiple of four here
#pragma unroll
            for (int q4 = 0; q4 < (EC + 3) / 4; ++q4) {
                const float4 f = reinterpret_cast<const float4*>(src)[q4];
                v[(4 * q4) % EC] = f.x;
                v[(4 * q4 + 1) % EC] = f.y;
                v[(4 * q4 + 2) % EC] = f.z;
                v[(4 * q4 + 3) % EC] = f.w;
            }
        } else {
#pragma unroll
            for (int q = 0; q < EC; ++q) {
                if (q < ec) v[q] = src[q];
            }
        }
    };
    // One lane = one channel of NY cells that follow each other in y.  For
    // every (dz, dy) the W weights of the tap row are read once and used by all
    // NY cells, and the NY tile rows they meet stay in registers from one dy to
    // the next (row dy + j serves cell j), so that a step costs one new tile
    // row and one weight row for NY * W fused multiply-adds.  Every cell still
    // sees its taps in table order: dz, then dy, then dx.
    constexpr int kNy = NY > 0 ? NY : 4;
    const int yq_n = G / kNy;
    const int combos = G * yq_n * G;
    auto window_sums = [&](const T* plane, const T* wq, T (&acc)[kNy]) {
#pragma unroll
        for (int j = 0; j < kNy; ++j) acc[j] = T(0);
#pragma unroll 1
        for (int dz = 0; dz < WT; ++dz) {
            const T* pz = plane + Tz * dz;
            T win[kNy][WT > 0 ? WT : 1];
#pragma unroll
            for (int yy = 0; yy < kNy - 1; ++yy) {
#pragma unroll
                for (int dx = 0; dx < WT; ++dx) win[yy][dx] = pz[Tn * yy + dx];
            }
#pragma unroll
            for (int dy = 0; dy < WT; ++dy) {
#pragma unroll
                for (int dx = 0; dx < WT; ++dx) {
                    win[(dy + kNy - 1) & (kNy - 1)][dx] = pz[Tn * (dy + kNy - 1) + dx];
                }
                T wr[WT > 0 ? WT : 1];
#pragma unroll
                for (int dx = 0; dx < WT; ++dx) wr[dx] = wq[(dz * WT + dy) * WT + dx];
#pragma unroll
                for (int j = 0; j < kNy; ++j) {
#pragma unroll
                    for (int dx = 0; dx < WT; ++dx) {
                        acc[j] = fma(win[(dy + j) & (kNy - 1)][dx], wr[dx], acc[j]);
                    }
                }
            }
        }
    };
    // Results go out through LDS when a thread can hold all of its items' sums
    // until the tile is no longer read: the tile's space then takes them cell
    // by cell (rows padded by one word against bank conflicts) and whole output
    // rows are written by consecutive lanes.  Written one channel per lane
    // straight from the registers, a row reaches memory as EC separate 4-byte
    // pieces from different wavefronts, which more than doubles the bytes
    // written.  Pays for its two barriers with full rows of 16 channels and
    // with 3^3 windows; the wider windows of narrower rows need the registers
    // that would hold the results for their window.
    constexpr int kHold = 4;
    const bool staged = YB && (EC >= 16 || (WT == 3 && EC >= 4)) && combos * EC <= kHold * kConvThreads;
    T held[kHold][kNy];
    // staged: combos divides the workgroup size, so the items of a thread are
    // the same cells in channels task_q, task_q + task_qstep, ...
    const int task_qstep = staged ? kConvThreads / combos : 0;
    const int task_q = staged ? tid / combos : EC;
    int task_plane = 0, task_cell = 0;
    if (staged) {
        const int rem = tid - task_q * combos;
        const int x = rem % G;
        const int y0 = kNy * ((rem / G) % yq_n);
        const int z = rem / (G * yq_n);
        task_plane = x + Tn * y0 + Tz * z;
        task_cell = (x + G * y0 + G * G * z) * (EC + 1);
    }
    int64_t blk = walk.next;
    int buf = 0;
    int64_t rows_reg = fetch_rows(blk);
    if (tid <= 27) s_nb[0][tid] = rows_reg;
    rows_reg = fetch_rows(blk + walk.step);
    __syncthreads();
    // what does not change from block to block is read once: the source and the
    // place in the tile of the rows this thread stages
    T pre[kPre][EC];
    uint32_t pre_src[kPre];
#pragma unroll
    for (int i = 0; i < kPre; ++i) {
        const int p = tid + i * kConvThreads;
        pre_src[i] = (prefetch && p < T3) ? s_src[p] : kNoRow;
    }
    if (prefetch) {
#pragma unroll
        for (int i = 0; i < kPre; ++i) load_row(s_nb[0], pre_src[i], pre[i]);
    }
    for (; blk < walk.end; blk += walk.step, buf ^= 1) {
        __syncthreads();  // the previous block's tile has been read
        const int64_t g = s_nb[buf][27];
        if (prefetch) {
#pragma unroll
            for (int i = 0; i < kPre; ++i) {
                if (pre_src[i] != kNoRow) {
                    T* at = tile + (pre_src[i] >> 17);
#pragma unroll
                    for (int q = 0; q < EC; ++q) at[YB ? q * Ts : q] = pre[i][q];
                }
            }
        } else {
            for (int p = tid; p < T3; p += kConvThreads) {
                T v[EC];
                const uint32_t src_cell = s_src[p];
                load_row(s_nb[buf], src_cell, v);
                T* at = tile + (src_cell >> 17);
#pragma unroll
                for (int q = 0; q < EC; ++q) at[YB ? q * Ts : q] = v[q];
            }
        }
        if (tid <= 27) s_nb[buf ^ 1][tid] = rows_reg;
        __syncthreads();
        rows_reg = fetch_rows(blk + 2 * walk.step);
        if (prefetch && blk + walk.step < walk.end) {
#pragma unroll
            for (int i = 0; i < kPre; ++i) load_row(s_nb[buf ^ 1], pre_src[i], pre[i]);
        }
        if (g < 0) continue;  // the same for the whole workgroup
        if constexpr (YB) {
            if (staged) {
#pragma unroll
                for (int it = 0; it < kHold; ++it) {
                    const int q = task_q + it * task_qstep;
                    if (q < ec) window_sums(tile + q * Ts + task_plane, s_w + q * K, held[it]);
                }
                __syncthreads();  // the tile has been read
                T* stage = tile;  // [M][EC + 1]
#pragma unroll
                for (int it = 0; it < kHold; ++it) {
                    const int q = task_q + it * task_qstep;
                    if (q >= ec) continue;
#pragma unroll
                    for (int j = 0; j < kNy; ++j) {
                        stage[task_cell + q + j * G * (EC + 1)] = held[it][j];
                    }
                }
                __syncthreads();
                T* out_g = out + static_cast<uint64_t>(static_cast<uint32_t>(g)) * block_words + e0;
                const uint8_t* mask_b = reinterpret_cast<const uint8_t*>(a.masks) + blk * a.M;
                if (vec && ec == EC) {   // whole rows, 16 bytes per lane
                    if constexpr (sizeof(T) == 4 && EC % 4 == 0) {
                        constexpr int kQ = EC / 4;
                        for (int i = tid; i < M * kQ; i += kConvThreads) {
                            const int c = i / kQ;
                            const int q4 = i - c * kQ;
                            const int c_i = s_inv[c];
                            const bool keep = c_i != 0xFFFF && mask_b[c_i];
                            if (!keep && !a.owns) continue;
                            const T* sp = stage + c * (EC + 1) + 4 * q4;
                            reinterpret_cast<float4*>(out_g + static_cast<uint32_t>(c) * E)[q4] =
                                    keep ? make_float4(sp[0], sp[1], sp[2], sp[3])
                                         : make_float4(0.f, 0.f, 0.f, 0.f);
                        }
                    }
                } else {
                    for (int i = tid; i < M * ec; i += kConvThreads) {
                        const int c = i / ec;
                        const int q = i - c * ec;
                        const int c_i = s_inv[c];
                        const bool keep = c_i != 0xFFFF && mask_b[c_i];
                        if (!keep && !a.owns) continue;
                        out_g[static_cast<uint32_t>(c) * E + q] = keep ? stage[c * (EC + 1) + q] : T(0);
                    }
                }
            } else {
#pragma unroll 1
                for (int at = tid; at < combos * EC; at += kConvThreads) {
                    const int q = at / combos;
                    if (q >= ec) continue;
                    const int rem = at - q * combos;
                    const int x = rem % G;
                    const int y0 = kNy * ((rem / G) % yq_n);
                    const int z = rem / (G * yq_n);
                    T acc[kNy];
                    window_sums(tile + static_cast<size_t>(q) * Ts + x + Tn * y0 + Tz * z,
                                s_w + static_cast<size_t>(q) * K, acc);
#pragma unroll
                    for (int j = 0; j < kNy; ++j) {
                        const int c = x + G * (y0 + j) + G * G * z;
                        const int c_i = s_inv[c];
                        const bool keep = c_i != 0xFFFF && a.masks[blk * a.M + c_i];
                        if (!keep && !a.owns) continue;
                        out[(g * a.M + c) * E + e0 + q] = keep ? acc[j] : T(0);
                    }
                }
            }
            continue;
        }
        clear_block(g);
        for (int c_i = tid; c_i < M; c_i += kConvThreads) {
            if (!a.masks[blk * a.M + c_i]) continue;
            const int64_t c64 = a.cell_indices[c_i];
            if (c64 < 0 || c64 >= a.M) continue;
            const int c = static_cast<int>(c64);
            // tile index of the tap (-r, -r, -r) of this cell
            const int base = c % G + Tn * ((c / G) % G) + Tn * Tn * (c / (G * G));
            T acc[EC];
#pragma unroll
            for (int q = 0; q < EC; ++q) acc[q] = T(0);
            // only the innermost loop is unrolled: a fully unrolled window keeps
            // hundreds of values in flight and costs the occupancy
#pragma unroll 1
            for (int dz = 0; dz < W; ++dz) {
#pragma unroll 1
                for (int dy = 0; dy < W; ++dy) {
                    const T* row = tile + static_cast<size_t>(base + Tn * dy + Tn * Tn * dz) * EC;
                    const T* wrow = s_w + static_cast<size_t>((dz * W + dy) * W) * EC;
                    if constexpr (WT > 0) {
#pragma unroll
                        for (int dx = 0; dx < WT; ++dx) {
#pragma unroll
                            for (int q = 0; q < EC; ++q) {
                                acc[q] = fma(row[dx * EC + q], wrow[dx * EC + q], acc[q]);
                            }
                        }
                    } else {
                        for (int dx = 0; dx < W; ++dx) {
#pragma unroll
                            for (int q = 0; q < EC; ++q) {
                                acc[q] = fma(row[dx * EC + q], wrow[dx * EC + q], acc[q]);
                            }
                        }
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < EC; ++q) {
                if (q < ec) out[(g * a.M + c) * E + e0 + q] = acc[q];
            }
        }
    }
}

// Settings of the tile kernel, each the fastest of the variants measured on
// 200 k blocks of 8^3 cells: windows from 27 taps on take the tile kernel, a
// tile may take 64 KB of LDS (two workgroups per CU), a lane handles four cells
// that follow each other in y (eight for windows of 5 and 7).
constexpr int kTileMinTaps = 27;
constexpr size_t kConvTileBytes = 64 * 1024;
constexpr bool kConvRowBlocking = true;
constexpr bool kConvRows8 = true;

// Largest cube edge G with G^3 == m, or 0.
inline int cube_edge(int64_t m) {
    int g = 1;
    while (static_cast<int64_t>(g) * g * g < m) ++g;
    return static_cast<int64_t>(g) * g * g == m ? g : 0;
}

// Takes the tile kernel when the sizes describe a cube window over cubic
// blocks with 27 neighbour blocks and the tile fits; returns -1 when not.
// `probe`: only say whether the tile kernel would take these sizes.
template <typename T>
int launch_convolution_tile(const ConvDev& a, hipStream_t s, bool probe = false) {
    const int G = cube_edge(a.M);
    const int W = cube_edge(a.K);
    if (G == 0 || W < 3 || W % 2 == 0 || a.GN != 27 || a.n_grids < 64) return -1;
    const int r = W / 2;
    if (r > G || a.M > 4096 || a.M * a.K > (int64_t{1} << 30)) return -1;
    const int64_t Tn = G + 2 * r;
    // cells per lane along y, as by_window below picks the instance
    const bool windowed = W == 3 || W == 5 || W == 7;
    const int ny = !(windowed && G % 4 == 0 && kConvRowBlocking) ? 0
                   : (G % 8 == 0 && kConvRows8 && W != 3) ? 8 : 4;
    // Words between the z layers of a channel's plane.  With blocks of 8^3 a
    // wavefront's lanes read 8 words along x per group, groups ny * Tn words
    // apart in y (four cells per lane) and one layer apart in z; the layers are
    // padded so that the four groups of every 32 lanes meet different banks.
    int64_t Tz = Tn * Tn;
    if (G == 8 && ny > 0 && sizeof(T) == 4) {
        const int a_y = static_cast<int>((4 * Tn) % 32);   // 8, 16 or 24
        int best = 32;
        for (int target : {8, 16, 24}) {
            const bool ok = ny == 8 ? target != 16 : (a_y == 16 ? target != 16 : target == 16);
            const int pad = static_cast<int>(((target - Tz) % 32 + 32) % 32);
            if (ok && pad < best) best = pad;
        }
        Tz += best;
    }
    // As many channels per pass as fit: a pass fetches the cache lines of all
    // channels of a row whatever it uses of them.
    constexpr int kMaxEc = sizeof(T) == 4 ? 16 : 8;
    const size_t cell_bytes = static_cast<size_t>(Tz * Tn) * sizeof(T);
    // two workgroups per CU (64 KB each) run faster than one with twice the
    // channels -- except for rows of a cache line or more, where every pass
    // over a part of the channels fetches the whole rows again: those may take
    // most of a CU's LDS for one workgroup (measured with 16 channels: 5^3
    // window in one pass 13.1 ms, in two passes of eight channels 15.5 ms)
    const size_t budget = a.E * sizeof(T) >= 64 ? 2 * kConvTileBytes : kConvTileBytes;
    int ec_max = kMaxEc;
    while (ec_max > 1 && cell_bytes * ec_max > budget) ec_max /= 2;
    if (cell_bytes * ec_max > budget) return -1;
    if (probe) return 0;
    const uintptr_t align = reinterpret_cast<uintptr_t>(a.in);
    for (int e0 = 0; e0 < a.E;) {
        int width = ec_max;                  // channels of the template instance
        while (width > 1 && width / 2 >= a.E - e0) width /= 2;
        const int ec = static_cast<int>(a.E - e0 < width ? a.E - e0 : width);
        const size_t smem = (cell_bytes + static_cast<size_t>(a.K) * sizeof(T)) * width +
                            static_cast<size_t>(Tn * Tn * Tn) * 4 + static_cast<size_t>(a.M) * 2 + 16;
        const int vec = (sizeof(T) == 4 && ec == width && width % 4 == 0 && a.E % 4 == 0 &&
                         e0 % 4 == 0 && align % 16 == 0) ? 1 : 0;
        const unsigned grid = persistent_grid(a.n_grids, smem + 512, 2048 / kConvThreads);
        auto launch = [&](auto kernel) -> int {
            ASH_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                        hipFuncAttributeMaxDynamicSharedMemorySize,
                                        static_cast<int>(smem)));
            kernel<<<grid, kConvThreads, smem, s>>>(a, G, r, e0, ec, vec, static_cast<int>(Tz));
            ASH_LAUNCH_CHECK();
            return 0;
        };
        auto by_window = [&](auto ec_tag) -> int {
            constexpr int kEc = decltype(ec_tag)::value;
            if (G % 4 == 0 && kConvRowBlocking) {
                if (G % 8 == 0 && kConvRows8) {
                    if (W == 5) return launch(convolution_tile_kernel<T, kEc, 5, 8>);
                    if (W == 7) return launch(convolution_tile_kernel<T, kEc, 7, 8>);
                }
                if (W == 3) return launch(convolution_tile_kernel<T, kEc, 3, 4>);
                if (W == 5) return launch(convolution_tile_kernel<T, kEc, 5, 4>);
                if (W == 7) return launch(convolution_tile_kernel<T, kEc, 7, 4>);
            }
            if (W == 3) return launch(convolution_tile_kernel<T, kEc, 3, 0>);
            if (W == 5) return launch(convolution_tile_kernel<T, kEc, 5, 0>);
            if (W == 7) return launch(convolution_tile_kernel<T, kEc, 7, 0>);
            return launch(convolution_tile_kernel<T, kEc, 0, 0>);
        };
        int rc = 1;
        if (width == 16) {
            if constexpr (kMaxEc >= 16) rc = by_window(std::integral_constant<int, 16>());
        } else if (width == 8) {
            rc = by_window(std::integral_constant<int, 8>());
        } else if (width == 4) {
            rc = by_window(std::integral_constant<int, 4>());
        } else if (width == 2) {
            rc = by_window(std::integral_constant<int, 2>());
        } else {
            rc = by_window(std::integral_constant<int, 1>());
        }
        if (rc) return 1;
        e0 += ec;
    }
    return 0;
}

template <typename T>
int launch_convolution_cells(const ConvDev& a, hipStream_t s) {
    const int64_t threads = a.n_grids * a.M;
    const int64_t blocks = (threads + kBlock - 1) / kBlock;
    if (blocks > 0x7FFFFFFFll) ASH_FAIL("convolution_forward: too many cells in one call");
    const unsigned gb = static_cast<unsigned>(blocks);
    const uintptr_t align = reinterpret_cast<uintptr_t>(a.in) | reinterpret_cast<uintptr_t>(a.out);
    const int vec4 = (sizeof(T) == 4 && a.E % 4 == 0 && align % 16 == 0) ? 1 : 0;
    if (a.K >= kTileMinTaps) {
        const int rc = launch_convolution_tile<T>(a, s);
        if (rc >= 0) return rc;
    }
    if (a.n_grids >= 64 && a.M <= 4096) {
        // enough blocks to keep persistent workgroups busy
        if (a.E <= 1) return launch_convolution_block<T, 1>(a, vec4, s);
        if (a.E <= 2) return launch_convolution_block<T, 2>(a, vec4, s);
        if (a.E <= 4) return launch_convolution_block<T, 4>(a, vec4, s);
        if (a.E <= 8) return launch_convolution_block<T, 8>(a, vec4, s);
        return launch_convolution_block<T, 16>(a, vec4, s);
    }
    if (a.E <= 1) {
        convolution_cell_kernel<T, 1><<<gb, kBlock, 0, s>>>(a, vec4);
    } else if (a.E <= 2) {
        convolution_cell_kernel<T, 2><<<gb, kBlock, 0, s>>>(a, vec4);
    } else if (a.E <= 4) {
        convolution_cell_kernel<T, 4><<<gb, kBlock, 0, s>>>(a, vec4);
    } else if (a.E <= 8) {
        convolution_cell_kernel<T, 8><<<gb, kBlock, 0, s>>>(a, vec4);
    } else {
        convolution_cell_kernel<T, 16><<<gb, kBlock, 0, s>>>(a, vec4);
    }
    ASH_LAUNCH_CHECK();
    return 0;
}

// Wider rows than the reference supports (its accumulator holds 16 channels):
// one lane per (cell, channel).
template <typename T>
__global__ __launch_bounds__(kBlock) void convolution_forward_kernel(ConvDev a) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    const int64_t item = t / a.E;
    const int e = static_cast<int>(t - item * a.E);
    if (item >= a.n_grids * a.M || !a.masks[item]) return;
    const int64_t g = a.grid_indices[item / a.M];
    const int64_t c = a.cell_indices[item % a.M];
    if (g < 0 || g >= a.B || c < 0 || c >= a.M) return;
    const T* in = static_cast<const T*>(a.in);
    const T* w = static_cast<const T*>(a.w);
    const int64_t* nb_g = a.lut_g + g * a.GN;
    const int64_t* nb_c = a.lut_c2c + c * a.K;
    const int64_t* nb_n = a.lut_c2g + c * a.K;
    T sum = T(0);
    for (int64_t k = 0; k < a.K; ++k) {
        const int64_t gn = nb_n[k];
        if (gn < 0 || gn >= a.GN) continue;
        const int64_t gi = nb_g[gn];
        if (gi < 0 || gi >= a.B) continue;
        const int64_t ci = nb_c[k];
        if (ci < 0 || ci >= a.M) continue;
        sum = fma(in[(gi * a.M + ci) * a.E + e], w[k * a.E + e], sum);
    }
    static_cast<T*>(a.out)[(g * a.M + c) * a.E + e] = sum;
}

__global__ __launch_bounds__(kBlock) void zero16_kernel(uint4* __restrict__ p,
                                                        int64_t n16) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock;
    const uint4 v = make_uint4(0u, 0u, 0u, 0u);
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
         i < n16; i += stride) {
        p[i] = v;
    }
}

__global__ __launch_bounds__(kBlock) void zero1_kernel(
        unsigned char* __restrict__ p, int64_t n) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
         i < n; i += stride) {
        p[i] = 0;
    }
}

// listed[b] = 1 for every block of the listing.
__global__ __launch_bounds__(kBlock) void mark_listed_kernel(
        const int64_t* __restrict__ grid_indices, int64_t n, int64_t B,
        uint8_t* __restrict__ listed) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    const int64_t g = grid_indices[i];
    if (g >= 0 && g < B) listed[g] = 1;
}

// Zeroes the rows of the blocks that are not listed: `units` 16-byte pieces
// per block, one workgroup per block at a time.
__global__ __launch_bounds__(kBlock) void zero_unlisted_kernel(
        uint4* __restrict__ out, const uint8_t* __restrict__ listed, int64_t B,
        int64_t units) {
    const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
    for (int64_t b = blockIdx.x; b < B; b += gridDim.x) {
        if (listed[b]) continue;  // the same for the whole workgroup
        uint4* rows = out + b * units;
        for (int64_t u = threadIdx.x; u < units; u += kBlock) rows[u] = zero;
    }
}

// ---------------------------------------------------------------- host
int zero_fill(void* ptr, int64_t bytes, hipStream_t s) {
    if (bytes <= 0) return 0;
    unsigned char* p = static_cast<unsigned char*>(ptr);
    // unaligned head
    const int64_t mis = (16 - reinterpret_cast<uintptr_t>(p) % 16) % 16;
    const int64_t head = mis < bytes ? mis : bytes;
    if (head > 0) {
        zero1_kernel<<<1, kBlock, 0, s>>>(p, head);
        ASH_LAUNCH_CHECK();
    }
    const int64_t n16 = (bytes - head) / 16;
    if (n16 > 0) {
        // one store per thread: workgroups handed out one after the other walk
        // through memory in order (6.8 TB/s; 5.7 with 16 384 workgroups striding)
        int64_t g = (n16 + kBlock - 1) / kBlock;
        if (g > 0x7FFFFFFF) g = 0x7FFFFFFF;
        zero16_kernel<<<static_cast<unsigned>(g), kBlock, 0, s>>>(
                reinterpret_cast<uint4*>(p + head), n16);
        ASH_LAUNCH_CHECK();
    }
    const int64_t tail = bytes - head - n16 * 16;
    if (tail > 0) {
        zero1_kernel<<<1, kBlock, 0, s>>>(p + head + n16 * 16, tail);
        ASH_LAUNCH_CHECK();
    }
    return 0;
}

// Runs of consecutive queries of a wavefront that meet the same row are summed
// before the atomic (2.4x faster on ray-ordered samples, neutral on shuffled
// ones); the kernels keep the plain variant as a template parameter.
constexpr bool merge_enabled() { return true; }

// `from_positions`: the per-query operand arrays are not read (the fused front
// end works them out), so they may be NULL.
int check_args(const ash_query_args* a, QDev& d, bool from_positions = false) {
    if (a == nullptr) ASH_FAIL("null query arguments");
    if (a->num_queries < 0) ASH_FAIL("negative query count");
    if (a->num_embeddings < 1 || a->cells_per_grid < 1) {
        ASH_FAIL("embeddings must have at least one block and one cell");
    }
    if (a->embedding_dim < 1 || a->embedding_dim > 16) {
        ASH_FAIL("embedding_dim must be in 1..16");
    }
    if (a->interpolation != ASH_INTERP_LINEAR &&
        a->interpolation != ASH_INTERP_SMOOTH_STEP) {
        ASH_FAIL("Unknown interpolation functor");
    }
    if (a->dtype != ASH_F32 && a->dtype != ASH_F64) ASH_FAIL("unknown dtype");
    if (a->num_embeddings > 0x7FFFFFFFll ||
        a->num_embeddings * a->cells_per_grid >= 0xFFFFFFFFll) {
        ASH_FAIL("num_embeddings * cells_per_grid must stay below 2^32 - 1");
    }
    if (a->embeddings == nullptr || a->lut_grid_nb2grid_idx == nullptr ||
        a->lut_cell_nb2cell_idx == nullptr || a->lut_cell_nb2grid_nb == nullptr) {
        ASH_FAIL("null table pointer");
    }
    if (a->num_queries > 0 && !from_positions &&
        (a->offsets == nullptr || a->grid_indices == nullptr ||
         a->cell_indices == nullptr || a->masks == nullptr)) {
        ASH_FAIL("null query pointer");
    }
    d.emb = a->embeddings;
    d.off = a->offsets;
    d.gidx = a->grid_indices;
    d.cidx = a->cell_indices;
    d.mask = a->masks;
    d.lut_g = a->lut_grid_nb2grid_idx;
    d.lut_c2c = a->lut_cell_nb2cell_idx;
    d.lut_c2g = a->lut_cell_nb2grid_nb;
    d.N = a->num_queries;
    d.B = a->num_embeddings;
    d.M = a->cells_per_grid;
    d.E = static_cast<int>(a->embedding_dim);
    d.smooth = a->interpolation == ASH_INTERP_SMOOTH_STEP ? 1 : 0;
    d.merge = merge_enabled() ? 1 : 0;
    return 0;
}

int pow2_ceil(int v) {
    int p = 1;
    while (p < v) p <<= 1;
    return p;
}

size_t smem_bytes(const QDev& d, int lpq) {
    return table_offset(d, lpq, lut_in_lds(d));
}

template <typename T, int VEC, int LPQ>
int launch_forward(const QDev& d, void* out, hipStream_t s) {
    const size_t smem = smem_bytes(d, LPQ);
    const unsigned g = persistent_grid((d.N + kBlock - 1) / kBlock, smem, forward_waves(VEC, LPQ));
    if (lut_in_lds(d)) {
        query_forward_kernel<T, VEC, LPQ, true>
                <<<g, kBlock, smem, s>>>(d, static_cast<T*>(out));
    } else {
        query_forward_kernel<T, VEC, LPQ, false>
                <<<g, kBlock, smem, s>>>(d, static_cast<T*>(out));
    }
    ASH_LAUNCH_CHECK();
    return 0;
}

template <typename T, int VEC, int LPQ>
int launch_grid_forward(const QDev& d, const FrontDev& f, void* out, hipStream_t s) {
    const size_t smem = smem_bytes(d, LPQ);
    const unsigned g = persistent_grid((d.N + kBlock - 1) / kBlock, smem, forward_waves(VEC, LPQ));
    const bool aux = f.gidx_out != nullptr;
#define ASH_GF(L, A)                                                          \
    grid_forward_kernel<T, VEC, LPQ, L, A><<<g, kBlock, smem, s>>>(d, f, static_cast<T*>(out))
    if (lut_in_lds(d)) {
        if (aux) ASH_GF(true, true);
        else ASH_GF(true, false);
    } else {
        if (aux) ASH_GF(false, true);
        else ASH_GF(false, false);
    }
#undef ASH_GF
    ASH_LAUNCH_CHECK();
    return 0;
}

template <typename T, int LPQ>
int launch_bwd_fwd(const QDev& d, const void* z, void* ge, void* go, const Second& also,
                   hipStream_t s) {
    const size_t smem = smem_bytes(d, LPQ);
    const int out = gradients_wanted(ge, go, also);
    const unsigned g = persistent_grid((d.N + kBlock - 1) / kBlock, smem,
                                       backward_waves<T>(out));
#define ASH_BF(L, O)                                                          \
    query_backward_forward_kernel<T, LPQ, L, O><<<g, kBlock, smem, s>>>(      \
            d, static_cast<const T*>(z), static_cast<T*>(ge),                 \
            static_cast<T*>(go), static_cast<const T*>(also.gg),              \
            static_cast<const T*>(also.z))
    if (lut_in_lds(d)) {
        if (out == 7) ASH_BF(true, 7);
        else if (out == 5) ASH_BF(true, 5);
        else if (out == 3) ASH_BF(true, 3);
        else if (out == 1) ASH_BF(true, 1);
        else ASH_BF(true, 2);
    } else {
        if (out == 7) ASH_BF(false, 7);
        else if (out == 5) ASH_BF(false, 5);
        else if (out == 3) ASH_BF(false, 3);
        else if (out == 1) ASH_BF(false, 1);
        else ASH_BF(false, 2);
    }
#undef ASH_BF
    ASH_LAUNCH_CHECK();
    return 0;
}

template <typename T, int LPQ>
int launch_bwd_bwd(const QDev& d, const void* gg, const void* z, void* gz,
                   void* ge, hipStream_t s) {
    const size_t smem = smem_bytes(d, LPQ);
    const int out = (ge != nullptr ? 1 : 0) | (gz != nullptr ? 2 : 0);
    const unsigned g = persistent_grid((d.N + kBlock - 1) / kBlock, smem,
                                       backward_waves<T>(out));
#define ASH_BB(L, O)                                                          \
    query_backward_backward_kernel<T, LPQ, L, O><<<g, kBlock, smem, s>>>(     \
            d, static_cast<const T*>(gg), static_cast<const T*>(z),           \
            static_cast<T*>(gz), static_cast<T*>(ge))
    if (lut_in_lds(d)) {
        if (out == 3) ASH_BB(true, 3);
        else if (out == 1) ASH_BB(true, 1);
        else ASH_BB(true, 2);
    } else {
        if (out == 3) ASH_BB(false, 3);
        else if (out == 1) ASH_BB(false, 1);
        else ASH_BB(false, 2);
    }
#undef ASH_BB
    ASH_LAUNCH_CHECK();
    return 0;
}

// Whether a backward goes by the kernels that give a lane a whole query, in fp32 (`out`: bit
// 0 scatters to the embeddings).  Widths of their own: 1 to 8 channels (four on 16-byte
// aligned buffers) and 12, as fields of a distance, colours, weights or four of either have
// them; 9 to 11 and 13 to 15 channels are built for a lane per channel alone, as every width
// of its own takes 0.4 MB of device code.  Of 16 what scatters nothing (a pair of its rows is
// two lines anyway, and sixteen floats of two kinds and eight rows are more than the
// registers hold), of 1 what scatters (a lane per channel is one per query there).  By a lane
// per channel -> by rows, us, queries along rays | in no order:
//   gradient of the positions alone: 300 000 of 2 channels 8.8 -> 7.8 | 22.0 -> 23.0, 1 M 26.7
//     -> 24.0 | 69.1 -> 71.2; 1 M of 3 33.1 -> 25.1 | 83.5 -> 83.9, of 5 58.6 -> 30.9 | 108.7 ->
//     106.6, of 7 58.7 -> 30.2 | 117.2 -> 116.1, of 8 59.1 -> 30.0 | 104.2 -> 102.1; 660 000 of
//     12 84.1 -> 28.2 | 92.5 -> 86.1, of 16 84.6 -> 35.4 | 91.4 -> 84.4
//   grad_z alone: 300 000 of 2 9.5 -> 7.9 | 20.7 -> 22.4, 1 M 26.3 -> 23.4 | 69.0 -> 70.5; 1 M of
//     3 32.0 -> 25.2 | 84.0 -> 83.6, of 5 46.7 -> 29.0 | 106.9 -> 108.8, of 7 48.0 -> 32.2 | 116.5
//     -> 121.9, of 8 48.3 -> 32.0 | 105.1 -> 107.5; 660 000 of 12 53.5 -> 30.3 | 89.1 -> 86.0, of
//     16 54.6 -> 37.2 | 87.8 -> 85.8
//   both orders of the scatter with the positions' gradient: 1 M of 1 72 -> 39 | 394 -> 231, of
//     2 96 -> 51 | 383 -> 231, of 3 123 -> 63 | 436 -> 283, of 5 172 -> 85 | 479 -> 340, of 7 185
//     -> 105 | 522 -> 390, of 8 145 -> 109 | 388 -> 330; 660 000 of 12 178 -> 127 | 399 -> 324;
//     1000 of 5 18.4 -> 8.6
// (Gathers in no order are bound by the lines of the rows either way; of two channels, and
// grad_z of five to eight, they lose 2 - 8 % there, where a lane asks for a line each.)
// What a query gets is the same to the bit whatever else is asked for, and so by either
// kind: both add up a query's corners and channels in the same order (row_product).  (The
// two kinds of sixteen channels in a launch each: 500 000 in order 139 -> 137, in none 218 ->
// 272.)
// Below 98 304 queries rows of one and two channels go by a lane per channel,
// which is there all the same and has less to set up: 50 000 of one 7.2 | 9.5, 90 000 10.1 |
// 11.5, 131 000 14.2 | 10.9; 70 000 of two 10.7 | 12.0, 131 000 15.9 | 12.1.
constexpr int64_t kNarrowScatter = int64_t{3} << 15;

bool rows_by_lane(const QDev& d, int out, const void* p0, const void* p1, const void* p2) {
    if (d.E == 4) return aligned16(d.emb) && aligned16(p0) && aligned16(p1) && aligned16(p2);
    if (d.E <= 2) return d.N >= kNarrowScatter && (d.E == 2 || (out & 1) != 0);
    return d.E <= 8 || d.E == 12 || (d.E == 16 && (out & 1) == 0);
}

template <typename T>
int dispatch_forward(const QDev& d, void* out, hipStream_t s) {
    if constexpr (sizeof(T) == 4) {
        if (d.E % 4 == 0 && aligned16(d.emb) && aligned16(out)) {
            switch (d.E / 4) {
                case 1:
                    return launch_forward<float, 4, 1>(d, out, s);
                case 2:
                    return launch_forward<float, 4, 2>(d, out, s);
                default:
                    return launch_forward<float, 4, 4>(d, out, s);
            }
        }
    }
    if constexpr (sizeof(T) == 4) {
        // narrow rows that are not a multiple of four channels: one lane takes
        // the whole row (six channels: two lanes, three each), instead of one
        // lane per channel with a power of two of lanes per query
        switch (d.E) {
            case 2:
                return launch_forward<float, 2, 1>(d, out, s);
            case 3:
                return launch_forward<float, 3, 1>(d, out, s);
            case 5:
                return launch_forward<float, 5, 1>(d, out, s);
            case 6:
                return launch_forward<float, 3, 2>(d, out, s);
            default:
                break;
        }
    }
    switch (pow2_ceil(d.E)) {
        case 1:
            return launch_forward<T, 1, 1>(d, out, s);
        case 2:
            return launch_forward<T, 1, 2>(d, out, s);
        case 4:
            return launch_forward<T, 1, 4>(d, out, s);
        case 8:
            return launch_forward<T, 1, 8>(d, out, s);
        default:
            return launch_forward<T, 1, 16>(d, out, s);
    }
}

// Same choice of variant as dispatch_forward, so that the fused kernel adds up
// the corner rows in the same order as ash_query_forward on the same operands.
template <typename T>
int dispatch_grid_forward(const QDev& d, const FrontDev& f, void* out, hipStream_t s) {
    if constexpr (sizeof(T) == 4) {
        if (d.E % 4 == 0 && aligned16(d.emb) && aligned16(out)) {
            switch (d.E / 4) {
                case 1:
                    return launch_grid_forward<float, 4, 1>(d, f, out, s);
                case 2:
                    return launch_grid_forward<float, 4, 2>(d, f, out, s);
                default:
                    return launch_grid_forward<float, 4, 4>(d, f, out, s);
            }
        }
    }
    if constexpr (sizeof(T) == 4) {
        // narrow rows that are not a multiple of four channels: one lane takes
        // the whole row (six channels: two lanes, three each), instead of one
        // lane per channel with a power of two of lanes per query
        switch (d.E) {
            case 2:
                return launch_grid_forward<float, 2, 1>(d, f, out, s);
            case 3:
                return launch_grid_forward<float, 3, 1>(d, f, out, s);
            case 5:
                return launch_grid_forward<float, 5, 1>(d, f, out, s);
            case 6:
                return launch_grid_forward<float, 3, 2>(d, f, out, s);
            default:
                break;
        }
    }
    switch (pow2_ceil(d.E)) {
        case 1:
            return launch_grid_forward<T, 1, 1>(d, f, out, s);
        case 2:
            return launch_grid_forward<T, 1, 2>(d, f, out, s);
        case 4:
            return launch_grid_forward<T, 1, 4>(d, f, out, s);
        case 8:
            return launch_grid_forward<T, 1, 8>(d, f, out, s);
        default:
            return launch_grid_forward<T, 1, 16>(d, f, out, s);
    }
}

template <typename T>
int dispatch_bwd_fwd(const QDev& d, const void* z, void* ge, void* go, const Second& also,
                     hipStream_t s) {
    if constexpr (sizeof(T) == 4) {
        const int out = gradients_wanted(ge, go, also);
        if (rows_by_lane(d, out, z, ge, also.z)) {
            switch (d.E) {
                case 1: return launch_bwd_fwd_vec<1>(d, z, ge, go, also, s);
                case 2: return launch_bwd_fwd_vec<2>(d, z, ge, go, also, s);
                case 3: return launch_bwd_fwd_vec<3>(d, z, ge, go, also, s);
                case 4: return launch_bwd_fwd_vec<4>(d, z, ge, go, also, s);
                case 5: return launch_bwd_fwd_vec<5>(d, z, ge, go, also, s);
                case 6: return launch_bwd_fwd_vec<6>(d, z, ge, go, also, s);
                case 7: return launch_bwd_fwd_vec<7>(d, z, ge, go, also, s);
                case 8: return launch_bwd_fwd_vec<8>(d, z, ge, go, also, s);
                case 12: return launch_bwd_fwd_vec<12>(d, z, ge, go, also, s);
                default: return launch_bwd_fwd_vec<16>(d, z, ge, go, also, s);
            }
        }
    }
    switch (pow2_ceil(d.E)) {
        case 1:
            return launch_bwd_fwd<T, 1>(d, z, ge, go, also, s);
        case 2:
            return launch_bwd_fwd<T, 2>(d, z, ge, go, also, s);
        case 4:
            return launch_bwd_fwd<T, 4>(d, z, ge, go, also, s);
        case 8:   // (fp32 rows of five to eight: all by rows)
            if constexpr (sizeof(T) == 8) return launch_bwd_fwd<T, 8>(d, z, ge, go, also, s);
            [[fallthrough]];
        default:
            return launch_bwd_fwd<T, 16>(d, z, ge, go, also, s);
    }
}

template <typename T>
int dispatch_bwd_bwd(const QDev& d, const void* gg, const void* z, void* gz,
                     void* ge, hipStream_t s) {
    if constexpr (sizeof(T) == 4) {
        const int out = (ge != nullptr ? 1 : 0) | (gz != nullptr ? 2 : 0);
        if (rows_by_lane(d, out, z, ge, gz)) {
            switch (d.E) {
                case 1: return launch_bwd_bwd_vec<1>(d, gg, z, gz, ge, s);
                case 2: return launch_bwd_bwd_vec<2>(d, gg, z, gz, ge, s);
                case 3: return launch_bwd_bwd_vec<3>(d, gg, z, gz, ge, s);
                case 4: return launch_bwd_bwd_vec<4>(d, gg, z, gz, ge, s);
                case 5: return launch_bwd_bwd_vec<5>(d, gg, z, gz, ge, s);
                case 6: return launch_bwd_bwd_vec<6>(d, gg, z, gz, ge, s);
                case 7: return launch_bwd_bwd_vec<7>(d, gg, z, gz, ge, s);
                case 8: return launch_bwd_bwd_vec<8>(d, gg, z, gz, ge, s);
                case 12: return launch_bwd_bwd_vec<12>(d, gg, z, gz, ge, s);
                default: return launch_bwd_bwd_vec<16>(d, gg, z, gz, ge, s);
            }
        }
    }
    switch (pow2_ceil(d.E)) {
        case 1:
            return launch_bwd_bwd<T, 1>(d, gg, z, gz, ge, s);
        case 2:
            return launch_bwd_bwd<T, 2>(d, gg, z, gz, ge, s);
        case 4:
            return launch_bwd_bwd<T, 4>(d, gg, z, gz, ge, s);
        case 8:   // (fp32 rows of five to eight: all by rows)
            if constexpr (sizeof(T) == 8) return launch_bwd_bwd<T, 8>(d, gg, z, gz, ge, s);
            [[fallthrough]];
        default:
            return launch_bwd_bwd<T, 16>(d, gg, z, gz, ge, s);
    }
}

int64_t elem_bytes(int dtype) { return dtype == ASH_F64 ? 8 : 4; }

}  // namespace
}  // namespace ash

using namespace ash;

extern "C" {

int ash_query_forward(const ash_query_args* a, void* output, void* stream) {
    QDev d;
    if (check_args(a, d)) return 1;
    if (d.N == 0) return 0;
    if (output == nullptr) ASH_FAIL("null output pointer");
    PointerGuard guard;
    ASH_HIP(guard.enter_for(a->embeddings));
    hipStream_t s = static_cast<hipStream_t>(stream);
    return a->dtype == ASH_F64 ? dispatch_forward<double>(d, output, s)
                               : dispatch_forward<float>(d, output, s);
}

int ash_grid_forward(ash_map_t* map, const float* x, const float* origin, float cell_size,
                     int grid_dim, const ash_query_args* tables, void* output, uint8_t* masks,
                     int64_t* grid_indices, int64_t* cell_indices, float* offsets,
                     void* stream) {
    if (map == nullptr) ASH_FAIL("null map handle");
    if (map->key_dim != 3) ASH_FAIL("grid queries need a map with 3-d keys");
    if (grid_dim < 1 || grid_dim > 1024) ASH_FAIL("grid_dim must be in 1..1024");
    if (!(cell_size > 0.f) || !(cell_size < INFINITY)) ASH_FAIL("cell_size must be positive and finite");
    QDev d;
    if (check_args(tables, d, true)) return 1;
    if (d.M != static_cast<int64_t>(grid_dim) * grid_dim * grid_dim) {
        ASH_FAIL("cells_per_grid must be grid_dim^3");
    }
    if (d.N > (int64_t{1} << 31) - kBlock) ASH_FAIL("too many positions in one call");
    if (d.N == 0) return 0;
    if (x == nullptr || output == nullptr || masks == nullptr) ASH_FAIL("null pointer");
    const int given = (grid_indices != nullptr) + (cell_indices != nullptr) + (offsets != nullptr);
    if (given != 0 && given != 3) {
        ASH_FAIL("grid_indices, cell_indices and offsets are written together: pass all or none");
    }
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (settle_table(map, s)) return 1;
    FrontDev f;
    f.m = map->d;
    f.x = x;
    f.origin = origin;
    f.inv_cell = 1.0f / cell_size;
    f.g = static_cast<float>(grid_dim);
    f.gdim = grid_dim;
    f.mask_out = masks;
    f.gidx_out = grid_indices;
    f.cidx_out = cell_indices;
    f.off_out = offsets;
    return tables->dtype == ASH_F64 ? dispatch_grid_forward<double>(d, f, output, s)
                                    : dispatch_grid_forward<float>(d, f, output, s);
}

namespace {

int backward_forward(const ash_query_args* a, const void* z, void* grad_embeddings,
                     void* grad_offsets, void* stream, bool clear, const Second& also = {},
                     double offset_scale = 1.0) {
    QDev d;
    if (check_args(a, d)) return 1;
    d.offset_scale = offset_scale;
    if (grad_embeddings == nullptr && grad_offsets == nullptr) {
        ASH_FAIL("at least one of grad_embeddings / grad_offsets is required");
    }
    PointerGuard guard;
    ASH_HIP(guard.enter_for(a->embeddings));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (clear && grad_embeddings != nullptr &&
        zero_fill(grad_embeddings, d.B * d.M * d.E * elem_bytes(a->dtype), s)) {
        return 1;
    }
    if (d.N == 0) return 0;
    if (z == nullptr) ASH_FAIL("null pointer");
    return a->dtype == ASH_F64
                   ? dispatch_bwd_fwd<double>(d, z, grad_embeddings,
                                              grad_offsets, also, s)
                   : dispatch_bwd_fwd<float>(d, z, grad_embeddings,
                                             grad_offsets, also, s);
}

int backward_backward(const ash_query_args* a, const void* grad_grad_offsets,
                      const void* z, void* grad_z, void* grad_embeddings,
                      void* stream, bool clear, double offset_scale = 1.0) {
    QDev d;
    if (check_args(a, d)) return 1;
    d.offset_scale = offset_scale;
    if (grad_embeddings == nullptr && grad_z == nullptr) {
        ASH_FAIL("at least one of grad_z / grad_embeddings is required");
    }
    PointerGuard guard;
    ASH_HIP(guard.enter_for(a->embeddings));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (clear && grad_embeddings != nullptr &&
        zero_fill(grad_embeddings, d.B * d.M * d.E * elem_bytes(a->dtype), s)) {
        return 1;
    }
    if (d.N == 0) return 0;
    if (z == nullptr || grad_grad_offsets == nullptr) ASH_FAIL("null pointer");
    return a->dtype == ASH_F64
                   ? dispatch_bwd_bwd<double>(d, grad_grad_offsets, z, grad_z,
                                              grad_embeddings, s)
                   : dispatch_bwd_bwd<float>(d, grad_grad_offsets, z, grad_z,
                                             grad_embeddings, s);
}

}  // namespace

int ash_query_backward_forward(const ash_query_args* a, const void* z,
                               void* grad_embeddings, void* grad_offsets,
                               void* stream) {
    return backward_forward(a, z, grad_embeddings, grad_offsets, stream, true);
}

int ash_query_backward_forward_accumulate(const ash_query_args* a, const void* z,
                                          void* grad_embeddings, void* grad_offsets,
                                          void* stream) {
    if (grad_embeddings == nullptr) ASH_FAIL("accumulate: null grad_embeddings");
    return backward_forward(a, z, grad_embeddings, grad_offsets, stream, false);
}

int ash_query_backward_both(const ash_query_args* a, const void* z, const void* grad_grad_offsets,
                            const void* z_second, void* grad_embeddings, void* grad_offsets,
                            int32_t accumulate, void* stream) {
    if (grad_embeddings == nullptr) ASH_FAIL("backward_both: null grad_embeddings");
    if (a != nullptr && a->num_queries > 0 && (grad_grad_offsets == nullptr || z_second == nullptr)) {
        ASH_FAIL("null pointer");
    }
    return backward_forward(a, z, grad_embeddings, grad_offsets, stream, accumulate == 0,
                            {grad_grad_offsets, z_second});
}

int ash_query_backward_backward(const ash_query_args* a,
                                const void* grad_grad_offsets, const void* z,
                                void* grad_z, void* grad_embeddings,
                                void* stream) {
    return backward_backward(a, grad_grad_offsets, z, grad_z, grad_embeddings, stream, true);
}

int ash_query_backward_backward_accumulate(const ash_query_args* a,
                                           const void* grad_grad_offsets, const void* z,
                                           void* grad_z, void* grad_embeddings,
                                           void* stream) {
    if (grad_embeddings == nullptr) ASH_FAIL("accumulate: null grad_embeddings");
    return backward_backward(a, grad_grad_offsets, z, grad_z, grad_embeddings, stream, false);
}

int ash_query_backward_forward_scaled(const ash_query_args* a, const void* z, const void* grad_grad_offsets,
                                      const void* z_second, void* grad_embeddings, void* grad_offsets,
                                      double offset_scale, int32_t accumulate, void* stream) {
    if (accumulate && grad_embeddings == nullptr) ASH_FAIL("accumulate: null grad_embeddings");
    if ((grad_grad_offsets == nullptr) != (z_second == nullptr)) ASH_FAIL("null pointer");
    if (grad_grad_offsets != nullptr && grad_embeddings == nullptr) {
        ASH_FAIL("backward_both: null grad_embeddings");
    }
    return backward_forward(a, z, grad_embeddings, grad_offsets, stream, accumulate == 0,
                            {grad_grad_offsets, z_second}, offset_scale);
}

int ash_query_backward_backward_scaled(const ash_query_args* a, const void* grad_grad_offsets,
                                       const void* z, void* grad_z, void* grad_embeddings,
                                       double offset_scale, int32_t accumulate, void* stream) {
    if (accumulate && grad_embeddings == nullptr) ASH_FAIL("accumulate: null grad_embeddings");
    return backward_backward(a, grad_grad_offsets, z, grad_z, grad_embeddings, stream, accumulate == 0,
                             offset_scale);
}

namespace {

int convolution_forward(const void* inputs, const void* weights,
                        const uint8_t* masks, const int64_t* grid_indices,
                        const int64_t* cell_indices,
                        const int64_t* lut_grid_nb2grid_idx,
                        const int64_t* lut_cell_nb2cell_idx,
                        const int64_t* lut_cell_nb2grid_nb, void* outputs,
                        int64_t num_grids, int64_t num_embeddings,
                        int64_t cells_per_grid, int64_t embedding_dim,
                        int64_t num_cell_nbs, int64_t num_grid_nbs,
                        int32_t dtype, uint8_t* listed, void* stream) {
    if (dtype != ASH_F32 && dtype != ASH_F64) ASH_FAIL("unknown dtype");
    if (num_grids < 0 || num_embeddings < 1 || cells_per_grid < 1 ||
        embedding_dim < 1 || num_cell_nbs < 1 || num_grid_nbs < 1) {
        ASH_FAIL("convolution_forward: bad sizes");
    }
    if (inputs == nullptr || weights == nullptr || outputs == nullptr ||
        lut_grid_nb2grid_idx == nullptr || lut_cell_nb2cell_idx == nullptr ||
        lut_cell_nb2grid_nb == nullptr) {
        ASH_FAIL("null pointer in convolution_forward");
    }
    if (num_grids > 0 && (masks == nullptr || grid_indices == nullptr ||
                          cell_indices == nullptr)) {
        ASH_FAIL("null pointer in convolution_forward");
    }
    PointerGuard guard;
    ASH_HIP(guard.enter_for(inputs));
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t scalar = dtype == ASH_F32 ? 4 : 8;
    ConvDev a;
    a.in = inputs;
    a.w = weights;
    a.masks = masks;
    a.grid_indices = grid_indices;
    a.cell_indices = cell_indices;
    a.lut_g = lut_grid_nb2grid_idx;
    a.lut_c2c = lut_cell_nb2cell_idx;
    a.lut_c2g = lut_cell_nb2grid_nb;
    a.out = outputs;
    a.n_grids = num_grids;
    a.B = num_embeddings;
    a.M = cells_per_grid;
    a.E = embedding_dim;
    a.K = num_cell_nbs;
    a.GN = num_grid_nbs;
    a.owns = 0;
    // Rows of blocks that are not listed stay zero (at::zeros_like,
    // grid.cu:1010).  With a scratch byte per block and the tile kernel, which
    // writes every cell of the blocks it is given, only those rows are cleared.
    const int64_t block_bytes = cells_per_grid * embedding_dim * scalar;
    const bool tile = num_grids > 0 && embedding_dim <= 16 && num_cell_nbs >= kTileMinTaps &&
                      (dtype == ASH_F32 ? launch_convolution_tile<float>(a, s, true)
                                        : launch_convolution_tile<double>(a, s, true)) == 0;
    if (listed != nullptr && tile && block_bytes % 16 == 0 &&
        reinterpret_cast<uintptr_t>(outputs) % 16 == 0) {
        if (zero_fill(listed, num_embeddings, s)) return 1;
        mark_listed_kernel<<<static_cast<unsigned>((num_grids + kBlock - 1) / kBlock), kBlock, 0,
                             s>>>(grid_indices, num_grids, num_embeddings, listed);
        ASH_LAUNCH_CHECK();
        const int64_t g = num_embeddings < 256 * 32 ? num_embeddings : 256 * 32;
        zero_unlisted_kernel<<<static_cast<unsigned>(g), kBlock, 0, s>>>(
                static_cast<uint4*>(outputs), listed, num_embeddings, block_bytes / 16);
        ASH_LAUNCH_CHECK();
        a.owns = 1;
    } else if (zero_fill(outputs, num_embeddings * block_bytes, s)) {
        return 1;
    }
    if (num_grids == 0) return 0;
    if (embedding_dim <= 16) {
        return dtype == ASH_F32 ? launch_convolution_cells<float>(a, s)
                                : launch_convolution_cells<double>(a, s);
    }
    const int64_t threads = num_grids * cells_per_grid * embedding_dim;
    const int64_t blocks = (threads + kBlock - 1) / kBlock;
    if (blocks > 0x7FFFFFFFll) ASH_FAIL("convolution_forward: too many cells in one call");
    if (dtype == ASH_F32) {
        convolution_forward_kernel<float><<<static_cast<unsigned>(blocks), kBlock, 0, s>>>(a);
    } else {
        convolution_forward_kernel<double><<<static_cast<unsigned>(blocks), kBlock, 0, s>>>(a);
    }
    ASH_LAUNCH_CHECK();
    return 0;
}

}  // namespace

int ash_convolution_forward(const void* inputs, const void* weights,
                            const uint8_t* masks, const int64_t* grid_indices,
                            const int64_t* cell_indices,
                            const int64_t* lut_grid_nb2grid_idx,
                            const int64_t* lut_cell_nb2cell_idx,
                            const int64_t* lut_cell_nb2grid_nb, void* outputs,
                            int64_t num_grids, int64_t num_embeddings,
                            int64_t cells_per_grid, int64_t embedding_dim,
                            int64_t num_cell_nbs, int64_t num_grid_nbs,
                            int32_t dtype, void* stream) {
    return convolution_forward(inputs, weights, masks, grid_indices, cell_indices,
                               lut_grid_nb2grid_idx, lut_cell_nb2cell_idx, lut_cell_nb2grid_nb,
                               outputs, num_grids, num_embeddings, cells_per_grid, embedding_dim,
                               num_cell_nbs, num_grid_nbs, dtype, nullptr, stream);
}

int ash_convolution_forward_listed(const void* inputs, const void* weights,
                                   const uint8_t* masks, const int64_t* grid_indices,
                                   const int64_t* cell_indices,
                                   const int64_t* lut_grid_nb2grid_idx,
                                   const int64_t* lut_cell_nb2cell_idx,
                                   const int64_t* lut_cell_nb2grid_nb, void* outputs,
                                   int64_t num_grids, int64_t num_embeddings,
                                   int64_t cells_per_grid, int64_t embedding_dim,
                                   int64_t num_cell_nbs, int64_t num_grid_nbs,
                                   int32_t dtype, uint8_t* listed, void* stream) {
    if (listed == nullptr) ASH_FAIL("convolution_forward_listed: null scratch");
    return convolution_forward(inputs, weights, masks, grid_indices, cell_indices,
                               lut_grid_nb2grid_idx, lut_cell_nb2cell_idx, lut_cell_nb2grid_nb,
                               outputs, num_grids, num_embeddings, cells_per_grid, embedding_dim,
                               num_cell_nbs, num_grid_nbs, dtype, listed, stream);
}

}  // extern "C"
