// Marching cubes over blocks of 8^3 cells in the layout the Python layer builds
// (cell c = x + 8 y + 64 z, neighbour b of the 2^3 window at bit pattern z y x):
// SparseDenseGrid.surface_mesh (ash/src/grid.cu:606-946 of the reference;
// ash_mesh.hip holds the kernels for other block sizes and for callers' tables).
//
// What the surface needs of a cell is two bits -- it weighs enough, it lies
// below the iso value -- so one pass over the field turns a block into 128
// bytes, and everything up to the vertex positions works on those:
//
//   bits     field and weights, read once and in memory order, wherever their values
//            lie in the rows (a channel of a wider tensor is not copied out
//            first): per block 8 + 8 words of 64 cells, a z layer each
//   classify a lane per row of eight cells along x: the cells the surface
//            crosses, their edges' owners and the number of their triangles,
//            eight cells at a time.  A row's three flag bytes (+x, +y, +z edge)
//            go to the block's own 64 words; what a block owes its neighbours
//            is at most nine 64-bit words, OR-ed into their face words
//   count    faces joined to the rows; where the points of a row start within
//            its block (8 bits from its layer, 16 from the block), where the
//            block's start within a group of 64
//   scan     running sums over the groups, totals to the host
//   points, triangles
//            a wavefront per block lists the block's points / triangles in LDS
//            and consecutive lanes handle consecutive ones.  A vertex id is the
//            start of the row plus the flags below the edge's.  One launch for both
//
// 60 000 blocks, field and weights in rows of five channels, us: listing 5, bits
// 98, classify 27, count and scan 20, points and triangles 99 (51 and 61 one after the
// other), together 249; with case bytes, a slot word per cell and the two channels copied
// out first: copies 274, clear, classify, count, points and triangles 415.
//
// Vertices are numbered along the listing, cells in order within a block, the
// axes in order within a cell, and triangles likewise: as in ash_mesh.hip.
#include "ash_table.h"
#include "ash_mc_table.h"
#include "ash_walk.h"

#include "../../include/ash_hip.h"

#include <functional>
#include <type_traits>

namespace ash {
namespace {

constexpr int kG = 8;
constexpr int kM = kG * kG * kG;
constexpr int kBlock = 256;
constexpr int kGroupBlocks = 64;      // blocks of the listing per running sum
constexpr int kCountThreads = 1024;
constexpr int kScanThreads = 1024;
constexpr int64_t kMaxStride = 64;
// One-wavefront workgroups of a walk over the blocks: several times what the
// device holds, because blocks differ in work (60 000 blocks, triangles / points /
// classify: 4096 workgroups 100 / 74 / 37 us, 8192 83 / 52 / 28, 16384 77 / 47 /
// 28, 65536 91 / 44 / 38, where setting up shows; with a lane per crossed cell and
// blocks fetched ahead 16384 55 / 48 / 25, 32768 55 / 46 / 28)
constexpr int kWalkGroups = 16384;
constexpr int kRoundCells = 192;      // crossed cells of a block whose triangles (up to five) are listed at a time
constexpr uint32_t kRowBits = 0x00FFFFFFu;
enum Face { kXy, kXz, kYx, kYz, kZx, kZy };   // face of the block, axis of the edges

struct Sums {
    int64_t points, triangles;
};

// The workspace: per row of the field tensor unless stated otherwise.
struct Work {
    uint64_t* bits;     // [B, 16]  bit x + 8 y of word z: weighs enough; of word 8 + z: below iso
    uint64_t* faces;    // [B, 8]   edges of the low-face cells that neighbours flag
    uint32_t* rows;     // [B, 64]  three flag bytes | points before in the layer << 24
    uint16_t* layer;    // [B, 8]   points before the layer in the block
    uint32_t* place;    // [B]      where the block stands in the listing (place_of)
    uint2* local;       // [n]      points and triangles before the listed block in its group
    Sums* groups;       // [ceil(n / kGroupBlocks)]
};

struct SurfaceArgs {
    const void* sdfs;
    const void* weights;
    const int64_t* grid_indices;
    const int32_t* grid_coords;   // [B, 3]
    const int64_t* lut_g;         // [B, 8]
    Work w;
    int64_t n, B;
    int64_t sdf_stride, weight_stride;   // elements between cells
    float iso, weight_thr;
    // world = cell * scale (+ origin), applied if `to_world`
    const float* origin;
    float scale;
    bool to_world;
    int64_t n_points, n_triangles;
    float* positions;
    int32_t* triangles;
};

int64_t groups_of(int64_t n) { return (n + kGroupBlocks - 1) / kGroupBlocks; }

int64_t align16(int64_t bytes) { return (bytes + 15) & ~int64_t{15}; }

int64_t lay_out(Work& w, char* base, int64_t n, int64_t B) {
    int64_t at = 0;
    auto take = [&](auto*& p, int64_t count) {
        p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(base + at);
        at += align16(count * static_cast<int64_t>(sizeof(*p)));
    };
    take(w.bits, 16 * B);
    take(w.faces, 8 * B);
    take(w.rows, 64 * B);
    take(w.layer, 8 * B);
    take(w.place, B);
    take(w.local, n);
    take(w.groups, groups_of(n));
    return at;
}

// Where the rows stand in the listing.  Rows that are not listed are not cleared (a
// launch less): whatever stands there, the listing does not name them at that place.
__global__ __launch_bounds__(kBlock) void place_listed_kernel(const int64_t* __restrict__ grid_indices,
                                                              int64_t n, int64_t B,
                                                              uint32_t* __restrict__ place) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    const int64_t g = grid_indices[i];
    if (g >= 0 && g < B) place[g] = static_cast<uint32_t>(i);
}

// The place of row g, or -1 where it is not listed: blocks that are not listed count
// as missing, their bits are zero.
__device__ __forceinline__ int64_t place_of(const SurfaceArgs& a, int64_t g) {
    const int64_t at = a.w.place[g];
    return at < a.n && a.grid_indices[at] == g ? at : -1;
}

// The bits of row g from the values of its cells, one layer per register: every
// lane of the wavefront calls this.
template <typename T>
__device__ __forceinline__ void leave_bits(const SurfaceArgs& a, int64_t g, const T (&v)[kG], const T (&w)[kG]) {
    const int lane = threadIdx.x & 63;
    uint64_t mine = 0;
#pragma unroll
    for (int z = 0; z < kG; ++z) {
        const uint64_t ok = __ballot(w[z] >= static_cast<T>(a.weight_thr));
        const uint64_t below = __ballot(v[z] - static_cast<T>(a.iso) < T(0));
        if (lane == z) mine = ok;
        if (lane == 8 + z) mine = below;
    }
    if (lane < 16) a.w.bits[g * 16 + lane] = mine;
    if (lane >= 16 && lane < 24) a.w.faces[g * 8 + (lane - 16)] = 0;
}

// One wavefront per row of the tensor, in memory order (blocks come in no order
// of memory in the listing: 60 000 rows of five channels 122 us along it, 107 in
// order), a lane per cell of a layer: sixteen loads in flight, the two values of
// a cell usually in one line.
template <typename T>
__global__ __launch_bounds__(kBlock) void bits_kernel(SurfaceArgs a) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t g = static_cast<int64_t>(blockIdx.x) * (kBlock / 64) + wave;
    if (g >= a.B) return;
    const auto nothing = [&] {
        if (lane < 16) a.w.bits[g * 16 + lane] = 0;
    };
    // (a place that may be the row's as a rule is: the rows are asked for along with the
    // listing)
    const int64_t at_most = a.w.place[g];
    if (at_most >= a.n) return nothing();
    const int64_t listed = a.grid_indices[at_most];
    const T* sdfs = static_cast<const T*>(a.sdfs) + g * kM * a.sdf_stride;
    const T* weights = static_cast<const T*>(a.weights) + g * kM * a.weight_stride;
    const int s = static_cast<int>(a.sdf_stride), t = static_cast<int>(a.weight_stride);
    T v[kG], w[kG];
#pragma unroll
    for (int z = 0; z < kG; ++z) {
        v[z] = sdfs[(z * 64 + lane) * s];
        w[z] = weights[(z * 64 + lane) * t];
    }
    if (listed != g) return nothing();
    leave_bits(a, g, v, w);
}

// The same where field and weights are two channels of rows of S: a block's rows
// come in whole, 16 bytes per lane and marked as not to be kept, and the two
// channels are picked in LDS.  Streams at what the device reads at most (7.1 TB/s,
// against 6.4 for loads that are kept): 60 000 rows of five channels 107 -> 98 us.
// `at`: the aligned start of row 0 of the tensor as far as the two channels go,
// `sdf`, `weight`: their places behind it.
template <int S>
__global__ __launch_bounds__(kBlock) void bits_staged_kernel(SurfaceArgs a, const float* at, int sdf, int weight) {
    typedef float v4 __attribute__((ext_vector_type(4)));
    __shared__ v4 s_rows[kBlock / 64][kM * S / 4];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t g = static_cast<int64_t>(blockIdx.x) * (kBlock / 64) + wave;
    if (g >= a.B) return;
    const auto nothing = [&] {
        if (lane < 16) a.w.bits[g * 16 + lane] = 0;
    };
    const int64_t at_most = a.w.place[g];   // (as above)
    if (at_most >= a.n) return nothing();
    const int64_t listed = a.grid_indices[at_most];
    // up to the last value that is needed: the rows may end with it
    const int pieces = ((kM - 1) * S + (sdf > weight ? sdf : weight)) / 4 + 1;
    const v4* rows = reinterpret_cast<const v4*>(at + g * (kM * S));
    v4 piece[2 * S];
#pragma unroll
    for (int i = 0; i < 2 * S; ++i) {
        const int p = i * 64 + lane;
        piece[i] = __builtin_nontemporal_load(rows + (p < pieces ? p : 0));
    }
    if (listed != g) return nothing();
#pragma unroll
    for (int i = 0; i < 2 * S; ++i) s_rows[wave][i * 64 + lane] = piece[i];
    // (a wavefront's own: its LDS instructions execute in order)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float* values = reinterpret_cast<const float*>(s_rows[wave]);
    float v[kG], w[kG];
#pragma unroll
    for (int z = 0; z < kG; ++z) {
        v[z] = values[(z * 64 + lane) * S + sdf];
        w[z] = values[(z * 64 + lane) * S + weight];
    }
    leave_bits(a, g, v, w);
}

// ------------------------------------------------------ a block and its corners
// The listing positions a one-wavefront workgroup walks, with what it needs of
// a block fetched one block (rows) and two blocks (index) ahead: lane l works
// for source s = l / 8, the block itself for s = 0, else neighbour s.
struct Blocks {
    const SurfaceArgs& a;
    TileWalk walk;
    int64_t at;         // listing position
    int64_t own, row;   // the block's row; the row of the lane's source, -1 if missing
    int64_t next_own, next_row, third_own;

    __device__ __forceinline__ int64_t index(int64_t b) const {
        if (b >= walk.end) return -1;
        const int64_t g = a.grid_indices[b];
        return (g >= 0 && g < a.B) ? g : -1;
    }
    __device__ __forceinline__ int64_t source(int64_t g) const {
        const int s = (threadIdx.x & 63) >> 3;
        if (g < 0) return -1;
        if (s == 0) return g;
        const int64_t r = a.lut_g[g * 8 + s];
        return (r >= 0 && r < a.B) ? r : -1;
    }
    __device__ __forceinline__ Blocks(const SurfaceArgs& args) : Blocks(args, blockIdx.x, gridDim.x) {}
    __device__ __forceinline__ Blocks(const SurfaceArgs& args, unsigned group, unsigned groups)
        : a(args), walk(args.n, group, groups), at(walk.next) {
        own = index(at);
        next_own = index(at + walk.step);
        row = source(own);
        third_own = index(at + 2 * walk.step);
        next_row = source(next_own);
    }
    __device__ __forceinline__ bool more() const { return at < walk.end; }
    // (the loads of `third_own` are waited for one block later)
    __device__ __forceinline__ void advance() {
        at += walk.step;
        own = next_own;
        row = next_row;
        next_own = third_own;
        third_own = index(at + 2 * walk.step);
        next_row = source(next_own);
    }
    // 16 of the 128 bytes of the lane's source, of this block and of the next
    __device__ __forceinline__ uint4 piece_of(int64_t r) const {
        if (r < 0) return make_uint4(0u, 0u, 0u, 0u);
        return reinterpret_cast<const uint4*>(a.w.bits + r * 16)[threadIdx.x & 7];
    }
    __device__ __forceinline__ uint4 piece() const { return piece_of(row); }
    __device__ __forceinline__ uint4 next_piece() const { return piece_of(next_row); }
};

// What lane (y, z) = (lane & 7, lane >> 3) knows of its row of cells: the bits
// "below" of the rows (y + dy, z + dz), nine cells long, in rows[dy + 2 dz], and
// the cells of the row (y, z) that the surface crosses.
struct RowCells {
    uint32_t below[4];
    uint32_t crossed;
};

// `bits`: the 128 bytes of the eight sources.
__device__ __forceinline__ RowCells row_cells(const uint8_t* bits) {
    const int lane = threadIdx.x & 63;
    RowCells r;
    uint32_t ok = 0xFFu, any = 0u, all = 0xFFu;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int y = (lane & 7) + (q & 1), z = (lane >> 3) + (q >> 1);
        const uint8_t* from = bits + (((y >> 3) << 1) | ((z >> 3) << 2)) * 128 + (y & 7) + 8 * (z & 7);
        const uint32_t o = from[0] | ((from[128] & 1u) << 8);
        const uint32_t b = from[64] | ((from[128 + 64] & 1u) << 8);
        ok &= o & (o >> 1);
        any |= b | (b >> 1);
        all &= b & (b >> 1);
        r.below[q] = b;
    }
    r.crossed = ok & any & ~all & 0xFFu;
    return r;
}

__device__ __forceinline__ uint32_t case_of(const RowCells& r, int x) {
    return ((r.below[0] >> x) & 3u) | (((r.below[1] >> x) & 3u) << 2) |
           (((r.below[2] >> x) & 3u) << 4) | (((r.below[3] >> x) & 3u) << 6);
}

__device__ __forceinline__ uint32_t lane_up(uint32_t v, int d) {
    return static_cast<uint32_t>(__shfl(static_cast<int>(v), ((threadIdx.x & 63) - d) & 63));
}

// The sum of the values of the lanes up to this one: every lane takes part, and no
// step goes through LDS (60 000 blocks, counts 18.3 -> 15.5 us, classify 26 -> 25).
template <int CTRL, int ROWS>
__device__ __forceinline__ int moved(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false);
}
__device__ __forceinline__ int sum_up_to(int v) {
    v += moved<0x111, 0xF>(v);   // lanes 1, 2, 4 and 8 before, of the row of 16
    v += moved<0x112, 0xF>(v);
    v += moved<0x114, 0xF>(v);
    v += moved<0x118, 0xF>(v);
    v += moved<0x142, 0xA>(v);   // the last lane of the row before
    v += moved<0x143, 0xC>(v);   // and of the lower half
    return v;
}
__device__ __forceinline__ int last_lane(int v) { return __builtin_amdgcn_readlane(v, 63); }

// Lists the crossed cells of a block in order, and the lanes' rows of "below" for
// case_at; returns their number.  What there is to do for a cell is then done by a
// lane per cell, some two rounds for a block; by a lane per row, each for its own
// cells, a round takes as many turns as the longest row has cells (five to eight;
// 60 000 blocks, 3.9 M triangles: 66 us, 54 this way).
__device__ __forceinline__ int list_crossed(const RowCells& r, uint2* rows, uint16_t* cells) {
    const int lane = threadIdx.x & 63;
    rows[lane] = make_uint2(r.below[0] | (r.below[1] << 16), r.below[2] | (r.below[3] << 16));
    const int own = __popc(r.crossed);
    const int upto = sum_up_to(own);
    const int row0 = (lane & 7) * kG + (lane >> 3) * 64;
    int at = upto - own;
    for (uint32_t left = r.crossed; left != 0u; left &= left - 1u) {
        cells[at++] = static_cast<uint16_t>(row0 + __builtin_ctz(left));
    }
    return last_lane(upto);
}
__device__ __forceinline__ uint32_t case_at(const uint2* rows, int cell) {
    const uint2 r = rows[cell >> 3];
    const uint32_t y0 = r.x >> (cell & 7), y1 = r.y >> (cell & 7);
    return (y0 & 3u) | ((y0 >> 14) & 12u) | ((y1 & 3u) << 4) | ((y1 >> 10) & 0xC0u);
}

__global__ __launch_bounds__(64) void classify_kernel(SurfaceArgs a) {
    __shared__ __align__(16) uint8_t s_bits[8 * 128];
    __shared__ uint8_t s_count[256];
    __shared__ __align__(8) uint8_t s_face[4 * 8];
    const int lane = threadIdx.x;
    const int y = lane & 7, z = lane >> 3;
    for (int i = lane; i < 256; i += 64) s_count[i] = static_cast<uint8_t>(kMcTriangleCount[i]);
    Blocks blk(a);
    uint4 piece = blk.piece();
    for (; blk.more(); blk.advance()) {
        __syncthreads();   // the previous block's bits and faces have been read
        reinterpret_cast<uint4*>(s_bits)[lane] = piece;
        __syncthreads();
        piece = blk.next_piece();   // on its way while this block is worked on
        const int64_t g = blk.own;
        if (g < 0) {   // the same for the whole wavefront
            if (lane == 0) a.w.local[blk.at] = make_uint2(0u, 0u);
            continue;
        }
        const RowCells r = row_cells(s_bits);
        if (__ballot(r.crossed != 0u) == 0) {
            a.w.rows[g * 64 + lane] = 0u;
            if (lane == 0) a.w.local[blk.at] = make_uint2(0u, 0u);
            continue;
        }
        // Crossed edges of the crossed cells, by the row of their owner: +x
        // edges of all four rows (eight bits), +y edges of the two rows at y,
        // +z edges of the two at z (nine bits: cell 8 belongs to the next block)
        const uint32_t c = r.crossed, c9 = c | (c << 1);
        uint32_t ex[4], ey[2], ez[2];
#pragma unroll
        for (int q = 0; q < 4; ++q) ex[q] = c & (r.below[q] ^ (r.below[q] >> 1));
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            ey[d] = c9 & (r.below[2 * d] ^ r.below[2 * d + 1]);
            ez[d] = c9 & (r.below[d] ^ r.below[d + 2]);
        }
        const uint32_t here = ex[0] | ((ey[0] & 0xFFu) << 8) | ((ez[0] & 0xFFu) << 16);
        const uint32_t corner = ex[3];
        uint32_t to_y = ex[1] | ((ez[1] & 0xFFu) << 16);
        uint32_t to_z = ex[2] | ((ey[1] & 0xFFu) << 8);
        const uint32_t from_z = lane_up(to_z, 8);
        if (const uint32_t up = lane_up(corner, 8); z > 0) to_y |= up;
        if (const uint32_t up = lane_up(corner, 1); y > 0) to_z |= up;
        uint32_t own = here;
        if (const uint32_t up = lane_up(to_y, 1); y > 0) own |= up;
        if (z > 0) own |= from_z;
        a.w.rows[g * 64 + lane] = own;

        if (y == 7) {
            s_face[z] = static_cast<uint8_t>(to_y);
            s_face[8 + z] = static_cast<uint8_t>(to_y >> 16);
        }
        if (z == 7) {
            s_face[16 + y] = static_cast<uint8_t>(to_z);
            s_face[24 + y] = static_cast<uint8_t>(to_z >> 8);
        }
        __syncthreads();
        const uint64_t y0 = __ballot(ey[0] >> 8), y1 = __ballot(ey[1] >> 8);   // by row
        const uint64_t z0 = __ballot(ez[0] >> 8), z1 = __ballot(ez[1] >> 8);
        constexpr uint64_t kLowY = 0x0101010101010101ull;
        uint64_t owed = 0;
        int to = 0, face = 0;
        auto owe = [&](int l, int s, int f, uint64_t word) {
            if (lane == l) {
                owed = word;
                to = s;
                face = f;
            }
        };
        const uint64_t* faces = reinterpret_cast<const uint64_t*>(s_face);
        owe(0, 1, kXy, y0 | (y1 << 8));
        owe(1, 1, kXz, z0 | ((z1 & ~(kLowY << 7)) << 1));
        owe(2, 2, kYx, faces[0]);
        owe(3, 2, kYz, faces[1]);
        owe(4, 4, kZx, faces[2]);
        owe(5, 4, kZy, faces[3]);
        owe(6, 5, kXy, y1 >> 56);
        owe(7, 3, kXz, (z1 >> 7) & kLowY);
        owe(8, 6, kYx, static_cast<uint32_t>(__builtin_amdgcn_readlane(corner, 63)));
        const int64_t dest = __shfl(blk.row, to * 8);
        if (owed != 0 && dest >= 0) {
            atomicOr(reinterpret_cast<unsigned long long*>(a.w.faces + dest * 8 + face),
                     static_cast<unsigned long long>(owed));
        }

        int triangles = 0;
        for (uint32_t left = c; left != 0u; left &= left - 1u) {
            triangles += s_count[case_of(r, __builtin_ctz(left))];
        }
        triangles = last_lane(sum_up_to(triangles));
        if (lane == 0) a.w.local[blk.at] = make_uint2(0u, static_cast<uint32_t>(triangles));
    }
}

// Sixteen wavefronts, four blocks each: the 64 blocks of a group.
__global__ __launch_bounds__(kCountThreads) void count_kernel(SurfaceArgs a) {
    constexpr int kEach = kGroupBlocks / (kCountThreads / 64);
    __shared__ int s_points[kGroupBlocks];
    const int lane = threadIdx.x & 63;
    // (the same for the whole wavefront: the faces come through the scalar cache)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int y = lane & 7, z = lane >> 3;
    const int64_t b0 = static_cast<int64_t>(blockIdx.x) * kGroupBlocks;
    int64_t g[kEach];
    uint32_t w[kEach];
    uint64_t face[kEach][6];
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const int64_t b = b0 + wave * kEach + k;
        g[k] = b < a.n ? a.grid_indices[b] : -1;
        if (g[k] >= a.B) g[k] = -1;
    }
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        w[k] = g[k] < 0 ? 0u : a.w.rows[g[k] * 64 + lane];
#pragma unroll
        for (int f = 0; f < 6; ++f) face[k][f] = g[k] < 0 ? 0u : a.w.faces[g[k] * 8 + f];
    }
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const auto byte = [&](int f, int i) { return static_cast<uint32_t>(face[k][f] >> (8 * i)) & 0xFFu; };
        w[k] |= (static_cast<uint32_t>(face[k][kXy] >> lane) & 1u) << 8;
        w[k] |= (static_cast<uint32_t>(face[k][kXz] >> lane) & 1u) << 16;
        if (y == 0) w[k] |= byte(kYx, z) | (byte(kYz, z) << 16);
        if (z == 0) w[k] |= byte(kZx, y) | (byte(kZy, y) << 8);
        const int own = __popc(w[k]);
        const int incl = sum_up_to(own);
        const int before = incl - own;
        const int layer = __shfl(before, lane & ~7);
        if (g[k] >= 0) {
            a.w.rows[g[k] * 64 + lane] = w[k] | (static_cast<uint32_t>(before - layer) << 24);
            if (y == 0) a.w.layer[g[k] * 8 + z] = static_cast<uint16_t>(layer);
        }
        if (lane == 63) s_points[wave * kEach + k] = incl;
    }
    __syncthreads();
    if (wave == 0) {
        const int64_t b = b0 + lane;
        const int points = s_points[lane];
        const int triangles = b < a.n ? static_cast<int>(a.w.local[b].y) : 0;
        const int p = sum_up_to(points), t = sum_up_to(triangles);
        if (b < a.n) a.w.local[b] = make_uint2(p - points, t - triangles);
        if (lane == 63) a.w.groups[blockIdx.x] = {p, t};
    }
}

// Sums of the groups -> what lies before each; totals for the host.
__global__ __launch_bounds__(kScanThreads) void scan_groups_kernel(Sums* __restrict__ groups, int64_t n,
                                                                   uint64_t* landing, int32_t stamp) {
    __shared__ Sums s_part[kScanThreads / 64];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int64_t per = (n + kScanThreads - 1) / kScanThreads;
    const int64_t first = threadIdx.x * per < n ? threadIdx.x * per : n;
    const int64_t last = first + per < n ? first + per : n;
    Sums mine = {0, 0};
    for (int64_t i = first; i < last; ++i) {
        mine.points += groups[i].points;
        mine.triangles += groups[i].triangles;
    }
    Sums incl = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int64_t up = __shfl_up(incl.points, d), ut = __shfl_up(incl.triangles, d);
        if (lane >= d) {
            incl.points += up;
            incl.triangles += ut;
        }
    }
    if (lane == 63) s_part[wave] = incl;
    __syncthreads();
    Sums before = {incl.points - mine.points, incl.triangles - mine.triangles}, total = {0, 0};
    for (int w = 0; w < kScanThreads / 64; ++w) {
        if (w < wave) {
            before.points += s_part[w].points;
            before.triangles += s_part[w].triangles;
        }
        total.points += s_part[w].points;
        total.triangles += s_part[w].triangles;
    }
    for (int64_t i = first; i < last; ++i) {
        const Sums own = groups[i];
        groups[i] = before;
        before.points += own.points;
        before.triangles += own.triangles;
    }
    if (threadIdx.x == 0) {
        const int32_t words[4] = {
                static_cast<int32_t>(total.points), static_cast<int32_t>(total.points >> 32),
                static_cast<int32_t>(total.triangles), static_cast<int32_t>(total.triangles >> 32)};
#pragma unroll
        for (int w = 0; w < 4; ++w) leave_word(landing + w, words[w], stamp);
    }
}

// Rounded twice, as the module's multiplication and addition are.
__device__ __forceinline__ float to_world(float p, float scale, const float* origin, int k) {
#pragma clang fp contract(off)
    const float scaled = p * scale;
    return origin == nullptr ? scaled : scaled + origin[k];
}

// The zero crossing of every flagged edge, linear between its two ends
// (ash/src/grid.cu:748-771).  Bound by the lines of the field that its cells and
// their partners lie in.
struct PointLists {
    uint16_t point[3 * kM];   // cell | axis << 9
};

template <typename T>
__device__ __forceinline__ void points_of(const SurfaceArgs& a, Blocks& blk, PointLists& lists) {
    uint16_t* const s_point = lists.point;
    const T* sdfs = static_cast<const T*>(a.sdfs);
    const int lane = threadIdx.x;
    const int row0 = (lane & 7) * kG + (lane >> 3) * 64;   // first cell of the lane's row
    // what the next block's list is made from is fetched while this one's points are
    uint32_t next_word = 0;
    int next_layer = 0;
    int64_t next_first = 0;
    auto fetch = [&](int64_t b, int64_t r) {
        if (r < 0) return;
        next_word = a.w.rows[r * 64 + lane];
        next_layer = a.w.layer[r * 8 + (lane >> 3)];
        next_first = a.w.groups[b / kGroupBlocks].points + a.w.local[b].x;
    };
    fetch(blk.at, blk.own);
    for (; blk.more(); blk.advance()) {
        const int64_t g = blk.own;
        const uint32_t word = next_word;
        int at = next_layer + static_cast<int>(word >> 24);
        const int64_t first = next_first;
        fetch(blk.at + blk.walk.step, blk.next_own);
        if (g < 0) continue;   // the same for the whole wavefront
        const uint32_t flags = word & kRowBits;
        if (__ballot(flags != 0u) == 0) continue;
        const int total = __shfl(at + __popc(flags), 63);
        __syncthreads();   // the previous block's list has been read
        for (uint32_t left = (flags | (flags >> 8) | (flags >> 16)) & 0xFFu; left != 0u; left &= left - 1u) {
            const int x = __builtin_ctz(left);
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                if ((flags >> (8 * d + x)) & 1u) s_point[at++] = static_cast<uint16_t>((row0 + x) | (d << 9));
            }
        }
        __syncthreads();
        const int32_t corner[3] = {a.grid_coords[g * 3] * kG, a.grid_coords[g * 3 + 1] * kG,
                                   a.grid_coords[g * 3 + 2] * kG};
        for (int q0 = 0; q0 < total; q0 += 64) {
            const int q = q0 + lane;
            const int entry = q < total ? s_point[q] : 0;
            const int cell = entry & (kM - 1);
            const int d = entry >> 9;
            const int shift = 3 * d;
            const int past = ((cell >> shift) & 7) == 7;
            // (all lanes take part: the row is that of another lane)
            const int64_t next = __shfl(blk.row, past ? 8 << d : 0);
            if (q >= total || first + q >= a.n_points) continue;   // (the latter never with the totals of the scan)
            const int partner = past ? cell & ~(7 << shift) : cell + (1 << shift);
            const T self = sdfs[(g * kM + cell) * a.sdf_stride] - static_cast<T>(a.iso);
            float ratio = 0.f;
            if (next >= 0) {
                const T other = sdfs[(next * kM + partner) * a.sdf_stride] - static_cast<T>(a.iso);
                ratio = static_cast<float>(self / (self - other));
            }
            float* out = a.positions + (first + q) * 3;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const float p = static_cast<float>(corner[k] + ((cell >> (3 * k)) & 7)) +
                                (d == k ? ratio : 0.f);
                out[k] = a.to_world ? to_world(p, a.scale, a.origin, k) : p;
            }
        }
    }
}

// Triangles of every crossed cell as ids of the points on its edges
// (ash/src/grid.cu:796-842); the table's rows have the orientation the reference
// writes.
struct TriangleLists {
    static constexpr int kRows = (kG + 1) * (kG + 1);
    __align__(16) uint8_t bits[8 * 128];        // of the eight sources; then the crossed cells
    uint2 rows[64];
    uint8_t case_of[kRoundCells];               // of the round's crossed cells
    uint16_t triangle[5 * kRoundCells];         // of the round: crossed cell | number in the cell << 8
    uint32_t flags[2 * kRows];                  // rows (y, z) of the block and of its +x neighbours
    uint32_t first[2 * kRows];
};

__device__ __forceinline__ void triangles_of(const SurfaceArgs& a, Blocks& blk, TriangleLists& lists) {
    constexpr int kRows = TriangleLists::kRows;
    uint8_t* const s_bits = lists.bits;
    uint8_t* const s_case = lists.case_of;
    uint2* const s_rows = lists.rows;
    uint16_t* const s_triangle = lists.triangle;
    uint16_t* const s_cell = reinterpret_cast<uint16_t*>(s_bits);   // (the bits are read by then)
    static_assert(sizeof(lists.bits) >= kM * sizeof(uint16_t), "all cells of a block");
    uint32_t* const s_flags = lists.flags;
    uint32_t* const s_first = lists.first;
    const int lane = threadIdx.x;
    // The first point of the lane's source, of this block and, a block ahead, of the next
    // (which is listed, or flags no edge).
    auto first_point = [&](int64_t place) {
        return place < 0 ? 0u : static_cast<uint32_t>(a.w.groups[place / kGroupBlocks].points) + a.w.local[place].x;
    };
    auto place = [&](int64_t r) { return r < 0 ? int64_t{-1} : place_of(a, r); };
    uint32_t source_first = first_point(place(blk.row));
    uint4 piece = blk.piece();
    for (; blk.more(); blk.advance()) {
        __syncthreads();   // the previous block's lists have been read
        reinterpret_cast<uint4*>(s_bits)[lane] = piece;
        __syncthreads();
        piece = blk.next_piece();   // on its way while this block is worked on
        const uint32_t starts = source_first;
        const int64_t next_place = place(blk.next_row);
        const RowCells r = row_cells(s_bits);
        source_first = first_point(next_place);
        if (blk.own < 0) continue;   // the same for the whole wavefront
        if (__ballot(r.crossed != 0u) == 0) continue;
        int64_t first = a.w.groups[blk.at / kGroupBlocks].triangles + a.w.local[blk.at].y;
#pragma unroll
        for (int k = 0; k < (2 * kRows + 63) / 64; ++k) {
            const int i = k * 64 + lane;
            const int side = i >= kRows, p = i - side * kRows;
            const int y = p % (kG + 1), z = p / (kG + 1);
            const int s = side | ((y >> 3) << 1) | ((z >> 3) << 2);
            const int64_t g = __shfl(blk.row, (s & 7) * 8);
            const uint32_t start = static_cast<uint32_t>(__shfl(static_cast<int>(starts), (s & 7) * 8));
            if (i >= 2 * kRows) continue;
            uint32_t word = 0, id = 0;
            if (g >= 0) {
                word = a.w.rows[g * 64 + (y & 7) + 8 * (z & 7)];
                id = start + a.w.layer[g * 8 + (z & 7)] + (word >> 24);
            }
            s_flags[i] = word & kRowBits;
            s_first[i] = id;
        }
        __syncthreads();   // the block's bits have been read
        const int crossed = list_crossed(r, s_rows, s_cell);
        __syncthreads();
        for (int c0 = 0; c0 < crossed; c0 += kRoundCells) {
            if (c0 > 0) __syncthreads();   // the previous round's list has been read
            int listed = 0;
            for (int c = c0; c < crossed && c < c0 + kRoundCells; c += 64) {
                const bool any = c + lane < crossed;
                const int at = c - c0 + lane;
                const uint32_t code = any ? case_at(s_rows, s_cell[c + lane]) : 0u;
                const int n = kMcTriangleCount[code];   // (none of case 0)
                if (any) s_case[at] = static_cast<uint8_t>(code);
                const int upto = sum_up_to(n);
                const int to = listed + upto - n;
#pragma unroll
                for (int t = 0; t < 5; ++t) {
                    if (t < n) s_triangle[to + t] = static_cast<uint16_t>(at | (t << 8));
                }
                listed += last_lane(upto);
            }
            __syncthreads();
            for (int q = lane; q < listed; q += 64) {
                if (first + q >= a.n_triangles) continue;   // never with the totals of the scan
                const int at = s_triangle[q] & 0xFF, t = s_triangle[q] >> 8;
                const int cell = s_cell[c0 + at];
                const uint32_t edges = static_cast<uint32_t>(kMcPackedRows[s_case[at]] >> (12 * t));
                const int x = cell & 7, y = (cell >> 3) & 7, z = cell >> 6;
                int32_t* out = a.triangles + (first + q) * 3;
#pragma unroll
                for (int v = 0; v < 3; ++v) {
                    // edge e = 4 axis + j starts at the corner made by a zero bit
                    // put into j at position `axis`
                    const int e = static_cast<int>(edges >> (4 * v)) & 15;
                    const int axis = e >> 2, j = e & 3;
                    const int low = (j & ((1 << axis) - 1)) | ((j >> axis) << (axis + 1));
                    const int px = x + (low & 1);
                    const int i = (px >> 3) * kRows + y + ((low >> 1) & 1) + (kG + 1) * (z + (low >> 2));
                    const uint32_t flags = s_flags[i];
                    const uint32_t before = ((1u << (px & 7)) - 1u) * 0x010101u;
                    const uint32_t lower = ((1u << (8 * axis)) - 1u) & (0x010101u << (px & 7));
                    out[v] = static_cast<int32_t>(s_first[i] + __popc(flags & (before | lower)));
                }
            }
            first += listed;
        }
    }
}

// Points and triangles by one launch, half of the workgroups each, of which every XCD has
// as many: the points wait for memory, the triangles for their vector instructions, and
// neither needs the other.  60 000 blocks of five channels, us: two launches 51 + 61, one
// 114 while the triangles kept their tables in LDS (7.6 KB a wavefront, 21 on a CU, of both
// kinds), 99 with the tables in the L1 and lists by round (4.9 KB, 28 on a CU); 27 000 of two
// channels 21 + 29 -> 42, 6000 of five 10 + 11 -> 15, 700 of two 7 + 7 -> 8.  Held to 64
// registers (32 on a CU) 102; lists of 128 cells instead of 192 101.
template <typename T>
__global__ __launch_bounds__(64) void extract_kernel(SurfaceArgs a) {
    __shared__ union {
        PointLists points;
        TriangleLists triangles;
    } s;
    const unsigned pair = blockIdx.x / (2 * kXcds), side = blockIdx.x / kXcds % 2;
    Blocks blk(a, pair * kXcds + blockIdx.x % kXcds, gridDim.x / 2);
    if (side == 0) points_of<T>(a, blk, s.points);
    else triangles_of(a, blk, s.triangles);
}

unsigned walk_grid(int64_t n) { return static_cast<unsigned>(n < kWalkGroups ? n : kWalkGroups); }

template <int S>
int launch_bits_staged(const SurfaceArgs& a, const float* at, int sdf, int weight, unsigned groups,
                       hipStream_t s) {
    bits_staged_kernel<S><<<groups, kBlock, 0, s>>>(a, at, sdf, weight);
    ASH_LAUNCH_CHECK();
    return 0;
}

// Two channels of the same rows, of two to eight channels and 16-byte
// aligned where the first of the two lies: through LDS.  (Wider rows would
// be read for the lines that neither channel lies in.)
int launch_bits(const SurfaceArgs& a, int32_t dtype, hipStream_t s) {
    const unsigned groups = static_cast<unsigned>((a.B + kBlock / 64 - 1) / (kBlock / 64));
    if (dtype == ASH_F64) {
        bits_kernel<double><<<groups, kBlock, 0, s>>>(a);
        ASH_LAUNCH_CHECK();
        return 0;
    }
    const float* sdfs = static_cast<const float*>(a.sdfs);
    const float* weights = static_cast<const float*>(a.weights);
    const float* at = std::less<const float*>()(sdfs, weights) ? sdfs : weights;
    const int64_t sdf = sdfs - at, weight = weights - at, stride = a.sdf_stride;
    if (a.weight_stride == stride && sdf < stride && weight < stride &&
        reinterpret_cast<uintptr_t>(at) % 16 == 0) {
        const int p = static_cast<int>(sdf), q = static_cast<int>(weight);
        switch (stride) {
            case 2: return launch_bits_staged<2>(a, at, p, q, groups, s);
            case 3: return launch_bits_staged<3>(a, at, p, q, groups, s);
            case 4: return launch_bits_staged<4>(a, at, p, q, groups, s);
            case 5: return launch_bits_staged<5>(a, at, p, q, groups, s);
            case 6: return launch_bits_staged<6>(a, at, p, q, groups, s);
            case 7: return launch_bits_staged<7>(a, at, p, q, groups, s);
            case 8: return launch_bits_staged<8>(a, at, p, q, groups, s);
            default: break;
        }
    }
    bits_kernel<float><<<groups, kBlock, 0, s>>>(a);
    ASH_LAUNCH_CHECK();
    return 0;
}

int fill(SurfaceArgs& a, const void* sdfs, int64_t sdf_stride, const int64_t* grid_indices,
         const int64_t* lut, int64_t n, int64_t B, float iso, int32_t dtype, void* workspace) {
    if (dtype != ASH_F32 && dtype != ASH_F64) ASH_FAIL("unknown dtype");
    if (n < 0 || B < 1 || n > (int64_t{1} << 31) || B > (int64_t{1} << 31)) {
        ASH_FAIL("surface extraction: bad sizes");
    }
    if (sdf_stride < 1 || sdf_stride > kMaxStride) ASH_FAIL("surface extraction: bad stride");
    if (n > 0 && (sdfs == nullptr || grid_indices == nullptr || lut == nullptr || workspace == nullptr)) {
        ASH_FAIL("null pointer in surface extraction");
    }
    if (reinterpret_cast<uintptr_t>(workspace) % 16 != 0) {
        ASH_FAIL("surface extraction: the workspace must be 16-byte aligned");
    }
    a.sdfs = sdfs;
    a.sdf_stride = sdf_stride;
    a.grid_indices = grid_indices;
    a.lut_g = lut;
    a.n = n;
    a.B = B;
    a.iso = iso;
    lay_out(a.w, static_cast<char*>(workspace), n, B);
    return 0;
}

}  // namespace
}  // namespace ash

using namespace ash;

extern "C" {

int64_t ash_surface_block8_workspace_bytes(int64_t num_grids, int64_t num_embeddings) {
    if (num_grids < 0 || num_embeddings < 1) return 0;
    Work w;
    return lay_out(w, nullptr, num_grids, num_embeddings);
}

int ash_surface_block8_classify(ash_map_t* map, const void* sdfs, int64_t sdf_stride,
                                const void* weights, int64_t weight_stride,
                                const int64_t* grid_indices, const int64_t* lut_grid_nb2grid_idx,
                                int64_t num_grids, int64_t num_embeddings, float iso_value,
                                float weight_thr, int32_t dtype, void* workspace, int64_t out[2],
                                void* stream) {
    if (map == nullptr) ASH_FAIL("null map handle");
    if (out == nullptr) ASH_FAIL("null output pointer");
    SurfaceArgs a = {};
    if (fill(a, sdfs, sdf_stride, grid_indices, lut_grid_nb2grid_idx, num_grids, num_embeddings,
             iso_value, dtype, workspace)) {
        return 1;
    }
    if (weight_stride < 1 || weight_stride > kMaxStride) ASH_FAIL("surface extraction: bad stride");
    out[0] = out[1] = 0;
    if (num_grids == 0) return 0;
    if (weights == nullptr) ASH_FAIL("null pointer in surface extraction");
    a.weights = weights;
    a.weight_stride = weight_stride;
    a.weight_thr = weight_thr;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (is_capturing(s)) {
        ASH_FAIL("the number of triangles cannot be read while the stream is being captured");
    }
    DeviceGuard guard;
    ASH_HIP(guard.enter(map->device));
    Answer answer;
    if (answer.take()) return 1;
    place_listed_kernel<<<static_cast<unsigned>((num_grids + kBlock - 1) / kBlock), kBlock, 0, s>>>(
            grid_indices, num_grids, num_embeddings, a.w.place);
    ASH_LAUNCH_CHECK();
    if (launch_bits(a, dtype, s)) return 1;
    classify_kernel<<<walk_grid(num_grids), 64, 0, s>>>(a);
    ASH_LAUNCH_CHECK();
    const int64_t groups = groups_of(num_grids);
    count_kernel<<<static_cast<unsigned>(groups), kCountThreads, 0, s>>>(a);
    ASH_LAUNCH_CHECK();
    scan_groups_kernel<<<1, kScanThreads, 0, s>>>(a.w.groups, groups, answer.words, answer.stamp);
    ASH_LAUNCH_CHECK();
    if (answer.wait(s, 4)) return 1;
    for (int w = 0; w < 2; ++w) out[w] = answer.pair(2 * w);
    if (out[0] > 0x7FFFFFFFll) ASH_FAIL("marching_cubes: more than 2^31 vertices");
    if (out[1] > 0x7FFFFFFFll / 3) ASH_FAIL("marching_cubes: too many triangles");
    return 0;
}

int ash_surface_block8_extract(const void* sdfs, int64_t sdf_stride, const int64_t* grid_indices,
                               const int32_t* grid_coords_table,
                               const int64_t* lut_grid_nb2grid_idx, int64_t num_grids,
                               int64_t num_embeddings, float iso_value, int32_t dtype,
                               void* workspace, int64_t n_vertices, int64_t n_triangles,
                               int to_world, float cell_to_world, const float* origin,
                               float* positions, int32_t* triangles, void* stream) {
    SurfaceArgs a = {};
    if (fill(a, sdfs, sdf_stride, grid_indices, lut_grid_nb2grid_idx, num_grids, num_embeddings,
             iso_value, dtype, workspace)) {
        return 1;
    }
    if (n_vertices < 0 || n_triangles < 0) ASH_FAIL("marching_cubes: negative counts");
    if (num_grids == 0 || n_vertices == 0) return 0;
    if (grid_coords_table == nullptr || positions == nullptr || (n_triangles > 0 && triangles == nullptr)) {
        ASH_FAIL("null pointer in marching_cubes");
    }
    a.grid_coords = grid_coords_table;
    a.to_world = to_world != 0;
    a.scale = cell_to_world;
    a.origin = origin;
    a.n_points = n_vertices;
    a.n_triangles = n_triangles;
    a.positions = positions;
    a.triangles = triangles;
    PointerGuard guard;
    ASH_HIP(guard.enter_for(sdfs));
    hipStream_t s = static_cast<hipStream_t>(stream);
    const unsigned groups = 2 * ((walk_grid(num_grids) + kXcds - 1) / kXcds * kXcds);
    auto kernel = dtype == ASH_F32 ? extract_kernel<float> : extract_kernel<double>;
    kernel<<<groups, 64, 0, s>>>(a);
    ASH_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
