// What the query kernels share (ash_query.hip, ash_rows.hip): operands, interpolation,
// tables of cells in LDS and the corner rows of a query.
#pragma once

#include "ash_probe.h"
#include "ash_walk.h"

#include <hip/amd_detail/amd_hip_unsafe_atomics.h>

#include "../../include/ash_hip.h"

namespace ash {

constexpr int kBlock = 256;
constexpr int64_t kMaxLdsCells = 2048;  // 2048 * 8 * 2 B = 32 KiB
constexpr uint32_t kNoRow = 0xFFFFFFFFu;
constexpr int kLdsPerCu = 160 * 1024;

struct QDev {
    const void* emb;
    const float* off;
    const int64_t* gidx;
    const int64_t* cidx;
    const uint8_t* mask;
    const int64_t* lut_g;
    const int64_t* lut_c2c;
    const int64_t* lut_c2g;
    int64_t N;
    int64_t B;
    int64_t M;
    int E;
    // Gradients with respect to the offsets are multiplied by it, both where they are
    // written and where the gradient of one is read: the grid's positions are offsets
    // in units of a cell, and a pass over the gradient behind or in front of the kernel
    // takes 17 - 23 us of 4 M queries (three of them in a training pass).
    double offset_scale = 1.0;
    int smooth;    // 0 linear, 1 smooth step
    int merge;     // pre-reduce runs of equal rows before the atomics
};

// Interpolation basis (ash/src/grid.cu:7-41).
template <typename T>
__device__ __forceinline__ T basis(T x, int smooth) {
    return smooth ? x * x * (T(3) - T(2) * x) : x;
}
template <typename T>
__device__ __forceinline__ T dbasis(T x, int smooth) {
    return smooth ? T(6) * x * (T(1) - x) : T(1);
}

// Per-axis factors of the corner weights and of their derivatives
// (ash/src/grid.cu:113-118,229-241): side 0 is the "1 - o" side.
template <typename T>
struct AxisTerms {
    T w[3][2];
    T dw[3][2];
};

template <typename T, bool GRAD>
__device__ __forceinline__ void axis_terms(const float (&o)[3], int smooth,
                                           AxisTerms<T>& t) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const T x1 = static_cast<T>(o[d]);
        const T x0 = static_cast<T>(1.0f - o[d]);
        t.w[d][0] = basis<T>(x0, smooth);
        t.w[d][1] = basis<T>(x1, smooth);
        if constexpr (GRAD) {
            t.dw[d][0] = -dbasis<T>(x0, smooth);
            t.dw[d][1] = dbasis<T>(x1, smooth);
        }
    }
}

template <typename T>
__device__ __forceinline__ T corner_weight(const AxisTerms<T>& t, int c) {
    T w = T(1);
    w *= t.w[0][c & 1];
    w *= t.w[1][(c >> 1) & 1];
    w *= t.w[2][(c >> 2) & 1];
    return w;
}

template <typename T>
__device__ __forceinline__ void corner_weight_grad(const AxisTerms<T>& t, int c,
                                                   T (&g)[3]) {
    const int b0 = c & 1, b1 = (c >> 1) & 1, b2 = (c >> 2) & 1;
    g[0] = t.dw[0][b0] * t.w[1][b1] * t.w[2][b2];
    g[1] = t.w[0][b0] * t.dw[1][b1] * t.w[2][b2];
    g[2] = t.w[0][b0] * t.w[1][b1] * t.dw[2][b2];
}

// grad w_c . u for the eight corners, with the products of the first two axes
// taken once for both sides of the third: half the operations of the sum of
// corner_weight_grad's three terms, and one rounding less on each.
template <typename T>
struct SlopeTerms {
    T w01[4], d01[4], d2[2];
};

template <typename T>
__device__ __forceinline__ void slope_terms(const AxisTerms<T>& t, const T (&u)[3], SlopeTerms<T>& s) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int b0 = i & 1, b1 = i >> 1;
        s.w01[i] = t.w[0][b0] * t.w[1][b1];
        s.d01[i] = (t.dw[0][b0] * u[0]) * t.w[1][b1] + t.w[0][b0] * (t.dw[1][b1] * u[1]);
    }
    s.d2[0] = t.dw[2][0] * u[2];
    s.d2[1] = t.dw[2][1] * u[2];
}

template <typename T>
__device__ __forceinline__ T corner_slope(const AxisTerms<T>& t, const SlopeTerms<T>& s, int c) {
    return s.d01[c & 3] * t.w[2][c >> 2] + s.w01[c & 3] * s.d2[c >> 2];
}

// ------------------------------------------------------------ LDS layout
// [ tile: row[8][256] uint32, off[3][256] float ]  (only when LPQ > 1)
// [ per-cell table: uint16[M][8] ]  (only when lds_lut)
// [ one LineTable per wavefront ]  (backward kernels by rows, ash_rows.hip, that produce grad_embeddings)
struct Tile {
    uint32_t row[8][kBlock];
    float off[3][kBlock];
};

// A cell's eight corners, one 16-bit code each (cell of the corner, below
// kMaxLdsCells, and number of its neighbour block above it): one 16-byte read
// per query.
struct CellLut {
    const uint4* codes;
};

constexpr int kCodeCellBits = 11;
static_assert(kMaxLdsCells == int64_t{1} << kCodeCellBits, "cells of a code");

template <bool LDS>
__device__ __forceinline__ void cell_neighbors(const QDev& a, const CellLut& lut, int64_t cell,
                                               uint32_t (&nb_cell)[8], uint32_t (&nb_grid)[8]) {
    if constexpr (LDS) {
        const uint4 v = lut.codes[cell];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const uint32_t code = (w[c >> 1] >> (16 * (c & 1))) & 0xFFFFu;
            nb_cell[c] = code & (kMaxLdsCells - 1);
            nb_grid[c] = code >> kCodeCellBits;
        }
    } else {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            int64_t v = a.lut_c2c[cell * 8 + c];
            v = v < 0 ? 0 : (v >= a.M ? a.M - 1 : v);
            nb_cell[c] = static_cast<uint32_t>(v);
            nb_grid[c] = static_cast<uint32_t>(a.lut_c2g[cell * 8 + c]) & 7u;
        }
    }
}

template <bool LDS, int THREADS = kBlock>
__device__ __forceinline__ CellLut stage_cell_lut(const QDev& a,
                                                  unsigned char* smem) {
    CellLut lut = {nullptr};
    if constexpr (LDS) {
        // a cell at a time: its sixteen table entries come by eight loads in flight
        uint4* codes = reinterpret_cast<uint4*>(smem);
        const int cells = static_cast<int>(a.M);
#pragma unroll 1
        for (int cell = threadIdx.x; cell < cells; cell += THREADS) {
            uint32_t nb_cell[8], nb_grid[8], w[4];
            cell_neighbors<false>(a, lut, cell, nb_cell, nb_grid);
#pragma unroll
            for (int c = 0; c < 8; c += 2) {
                w[c >> 1] = nb_cell[c] | (nb_grid[c] << kCodeCellBits) | (nb_cell[c + 1] << 16) |
                            (nb_grid[c + 1] << (16 + kCodeCellBits));
            }
            codes[cell] = make_uint4(w[0], w[1], w[2], w[3]);
        }
        __syncthreads();
        lut.codes = reinterpret_cast<const uint4*>(smem);
    }
    return lut;
}

// Where the line tables of the backward kernels by rows start in dynamic LDS.
__host__ __device__ inline size_t table_offset(const QDev& a, int lpq, bool lds_lut) {
    size_t bytes = lpq > 1 ? sizeof(Tile) : 0;
    if (lds_lut) bytes += static_cast<size_t>(a.M) * 8 * 2;
    return (bytes + 15) & ~static_cast<size_t>(15);
}

// What a query brings.  The mask, the indices and the offsets are asked for
// together (one trip to memory, not two); what a masked query has there is read
// and dropped.  They are read once, like z, and the per-query outputs are
// written once: those loads and stores carry the non-temporal hint, which
// leaves the caches to the embedding rows (forward, E = 4: 0.129 -> 0.117 ms).
struct QueryInputs {
    // low dwords of the int64 indices: a row of the block table is below 2^31
    // and "none" is -1, a cell is below 2^31 too
    int32_t gi, ci;
    float o[3];
    uint8_t m;   // 0: masked out or beyond the last query
};

__device__ __forceinline__ QueryInputs load_inputs(const QDev& a, int64_t q) {
    QueryInputs in;
    in.gi = in.ci = 0;
    in.o[0] = in.o[1] = in.o[2] = 0.f;
    in.m = 0;
    if (q < a.N) {
        in.m = __builtin_nontemporal_load(a.mask + q);
        in.gi = __builtin_nontemporal_load(reinterpret_cast<const int32_t*>(a.gidx) + q * 2);
        in.ci = __builtin_nontemporal_load(reinterpret_cast<const int32_t*>(a.cidx) + q * 2);
        in.o[0] = __builtin_nontemporal_load(a.off + q * 3 + 0);
        in.o[1] = __builtin_nontemporal_load(a.off + q * 3 + 1);
        in.o[2] = __builtin_nontemporal_load(a.off + q * 3 + 2);
    }
    return in;
}

// Phase 1 for one query: the 8 corner rows (kNoRow in row[0] when the query is
// masked out, out of range, or misses a neighbour block) and the offsets.
// Latency bounds it, so the eight table entries are asked for together and
// checked afterwards.  Leaving at the first missing corner made every entry wait
// for the one before it, up to eight trips to the L2 in nearly every wavefront
// (one of its lanes stands at a block's edge), and the branches kept 126 - 168
// registers alive instead of 53 - 94, three or four wavefronts per SIMD instead
// of five to eight.  2^22 ray samples, rows of four, 200 k blocks: forward with
// its operands 166 -> 131 us, gradient of the positions 158 -> 87, backward 296
// -> 219, second order 262 -> 212; 10^6 samples, rows of sixteen: 75 -> 56, 140
// -> 121, 293 -> 220, 200 -> 167.
template <bool LDS>
__device__ __forceinline__ void resolve_rows(const QDev& a, const CellLut& lut,
                                             const QueryInputs& in, uint32_t (&row)[8],
                                             float (&o)[3]) {
    bool valid = in.m != 0 && static_cast<uint32_t>(in.gi) < static_cast<uint32_t>(a.B);
    const int64_t gi = valid ? in.gi : 0;
#pragma unroll
    for (int d = 0; d < 3; ++d) o[d] = valid ? in.o[d] : 0.f;
    const int64_t ci = in.ci < 0 ? 0 : (in.ci >= a.M ? a.M - 1 : in.ci);
    // Block indices are below 2^31 and a missing block is -1, so the low
    // dword of each int64 table entry carries everything.
    const int32_t* lut_g32 = reinterpret_cast<const int32_t*>(a.lut_g) + gi * 16;
    uint32_t nb_cell[8], nb_grid[8];
    int32_t own = -1, other[8];
    if (valid) own = lut_g32[0];
    cell_neighbors<LDS>(a, lut, ci, nb_cell, nb_grid);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        other[c] = -1;
        if (valid && nb_grid[c] != 0) other[c] = lut_g32[nb_grid[c] * 2];
    }
    const uint32_t cells = static_cast<uint32_t>(a.M);
    uint32_t most = 0;   // a missing block is the largest number
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const uint32_t g = static_cast<uint32_t>(nb_grid[c] != 0 ? other[c] : own);
        most = g > most ? g : most;
        row[c] = g * cells + nb_cell[c];
    }
    valid = valid && most < static_cast<uint32_t>(a.B);
    if (!valid) row[0] = kNoRow;
}

template <bool LDS>
__device__ __forceinline__ void resolve_rows(const QDev& a, const CellLut& lut,
                                             int64_t q, uint32_t (&row)[8],
                                             float (&o)[3]) {
    resolve_rows<LDS>(a, lut, load_inputs(a, q), row, o);
}

// Rows of two, three or five fp32 channels taken whole by one lane: a row is
// only 4-byte aligned in general (rows of 12 or 20 bytes follow each other), which is
// all a global load of several dwords asks for on this device.
template <int N>
struct alignas(4) FloatRow {
    float v[N];
};
// ---------------------------------------------------------------- host
// Whether the per-cell tables go to LDS.  Up to 2^19 queries a workgroup of a
// full device meets one tile, and filling its LDS (sixteen table entries a cell,
// a trip to the L2 and a barrier) costs more than reading the tables where they
// are.  Blocks of 8^3, ray-ordered queries: forward of 131 k rows of four 7.5 ->
// 6.1 us, 524 k 23.5 -> 17.2; gradient of the positions 524 k 21.3 -> 14.3; rows
// of sixteen 131 k 9.8 -> 8.3.  Unordered ones, rows of four: 100 k 15.5 -> 14.3,
// 500 k 56.1 and 56.0.  Above, ordered and unordered queries part (1 M: 33.9
// against 27.1, and 109 against 117), and at 4 M LDS is ahead for both (132
// against 139, 701 against 745 for rows of sixteen).
constexpr int64_t kMaxDirectQueries = int64_t{1} << 19;
inline bool lut_in_lds(const QDev& d) { return d.M <= kMaxLdsCells && d.N > kMaxDirectQueries; }

// Enough persistent workgroups to fill every CU as far as LDS allows.
inline unsigned persistent_grid(int64_t ntiles, size_t smem, int max_per_cu = 8) {
    int per_cu = max_per_cu;
    if (smem > 0) {
        const int fit = static_cast<int>(kLdsPerCu / smem);
        if (fit < per_cu) per_cu = fit < 1 ? 1 : fit;
    }
    int64_t g = static_cast<int64_t>(compute_units()) * per_cu;
    if (g > ntiles) g = ntiles;
    g = (g + kXcds - 1) / kXcds * kXcds;  // whole rounds over the XCDs
    if (g < kXcds) g = kXcds;
    return static_cast<unsigned>(g);
}

// What a first-order backward takes along of the second order: nothing, or the
// gradient with respect to the offsets' gradient and the z of that pass.
struct Second {
    const void* gg;
    const void* z;
};

inline int gradients_wanted(const void* ge, const void* go, const Second& also) {
    return (ge != nullptr ? 1 : 0) | (go != nullptr ? 2 : 0) | (also.gg != nullptr ? 4 : 0);
}

inline bool aligned16(const void* p) {
    return reinterpret_cast<uintptr_t>(p) % 16 == 0;
}

// Backward and backward of the backward by rows of E floats (ash_rows.hip).
template <int E>
int launch_bwd_fwd_vec(const QDev& d, const void* z, void* ge, void* go, const Second& also, hipStream_t s);
template <int E>
int launch_bwd_bwd_vec(const QDev& d, const void* gg, const void* z, void* gz, void* ge, hipStream_t s);

}  // namespace ash
