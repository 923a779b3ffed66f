// Sparse convolution over blocks of 8^3 cells with a cube window, for rows of up
// to eight float32 channels: the case of SparseDenseGrid.convolution and
// gaussian_filter_ on the grids of the demos (ash/src/grid.cu:948-1043;
// ash_query.hip holds the kernels for every other shape).
//
// The layout is the one the Python layer builds (cell c = x + 8 y + 64 z; tap k =
// (dx + r) + W (dy + r) + W^2 (dz + r); neighbour block (bx + 1) + 3 (by + 1) + 9
// (bz + 1)), so no per-cell table is read, checked or needed.
//
// One or two wavefronts per channel (Shape::kOneEach), lane = (x, z), eight or
// four cells along y per lane: a row of the tile is read once for all cells that
// need it, and a tap's weight is one scalar for the wavefront.  Every cell still
// sees its taps in table order, one fused multiply-add per tap, as in the other
// kernels.
//
// 60 000 blocks, the kernel alone: five channels 3^3 321 us (345 with the halo word by
// word, its missing rows selected and the taps read lane by lane; 1275 with tables and
// instances for powers of two); 40 000 blocks of two 87 -> 74 us a call; 4000 blocks,
// 7^3, of five 215 -> 195.  3^3 windows of five channels move 1.61 GB beyond the L2s at
// 5.0 TB/s, what a large copy reaches, and are bound by that: 0.61 GB of results and
// 1.0 of rows, 1.6 times what there are (the halo along x takes most lines of two
// neighbours; the listing along other curves changes nothing).  Without any
// arithmetic 307 us, without the results' way out 220; vector instructions are issued
// in 0.47 of the cycles, the LDS is busy in 0.52.  7^3 windows are bound by vector
// instructions (of two channels in 0.87 of the cycles).
//
// A tile is kT * kT lines of eight cells along x, contiguous in memory whatever the
// width of the rows: they come in as 16-byte pieces, and results leave the same way,
// through LDS.  The lines' ends come word by word (consecutive lanes, consecutive
// words of a row).  Where a piece or word goes in the tile never changes from block to
// block and is kept in registers.  Software pipeline: while a block is computed the
// next block's pieces are on their way into registers and the row numbers of the one
// after are fetched.  Rows of missing blocks are staged as zeros (with finite weights
// adding 0 * w leaves a sum as it is).
#include "ash_table.h"
#include "ash_walk.h"

#include "../../include/ash_hip.h"

namespace ash {
namespace {

constexpr int kG = 8;
constexpr int kM = kG * kG * kG;
constexpr int kMaxChannels = 8;
constexpr int kFillBlock = 256;

template <int E, int W>
struct Shape {
    static constexpr int kR = W / 2;
    static constexpr int kT = kG + 2 * kR;
    // words between the z layers of a channel's plane: 8 or 24 modulo 32, so
    // that the four groups of lanes (eight words along x, one z each) that are
    // served together meet different banks
    static constexpr int layer() {
        int p = kT * kT;
        while (p % 32 != 8 && p % 32 != 24) ++p;
        return p;
    }
    static constexpr int kLayer = layer();
    // and between the planes of two channels: what makes the fewest lanes meet at a bank
    // where a block's rows are put into the tile, counted for each shape over the places
    // below (cycles of a block, without and with: five channels, 3^3, 382 -> 366, 5^3 1068
    // -> 570, 7^3 1445 -> 908; eight channels 600 -> 450, 1728 -> 720, 1960 -> 1078).
    static constexpr int plane_gap() {
        constexpr int kGap[3][8] = {{0, 0, 30, 8, 18, 4, 2, 4},
                                    {0, 16, 4, 8, 4, 4, 18, 4},
                                    {0, 0, 30, 8, 2, 2, 30, 4}};
        return kGap[kR - 1][E - 1];
    }
    static constexpr int kPlane = kLayer * kT + plane_gap();
    // results on their way out: a z layer's rows, some words apart from the next
    // layer's (banks: a wavefront writes a word of eight cells in eight layers, 16
    // cycles for eight of these with five channels and a gap of eight, 32 with four)
    static constexpr int kOutLayer = 64 * E + (E % 4 == 0 ? 4 : 8);
    static constexpr int kTileWords = E * kPlane;
    static constexpr int kOutWords = kG * kOutLayer;
    // The taps of a 3^3 window stay in scalar registers; those of the others are read
    // from LDS, a lane each, and handed out lane by lane (one instruction per tap).
    static constexpr bool kTapsHeld = W == 3;
    static constexpr int kWeightWords = kTapsHeld ? 0 : E * W * 64;
    static constexpr int kFit = 160 * 1024 / (4 * (kTileWords + kOutWords + kWeightWords) + 1024);
    // Cells along y per lane, and with them wavefronts per channel.  Two per
    // channel, but for odd numbers of channels, where that is no multiple of the
    // four SIMDs: a CU then takes fewer workgroups than its registers hold (five
    // channels, ten wavefronts of 64 registers: two, not three, and the third of
    // the grid ran behind, 16 wavefronts per CU on average).  There one wavefront
    // per channel, and helpers up to a multiple of four that only load and
    // store; where the LDS holds a single workgroup, two per channel are better.
    // 40 000 blocks, 3^3: three channels 101 -> 103 us, five 284 -> 208, seven
    // 355 -> 278; 12 000 blocks, 5^3: 139 -> 120, 218 -> 208, 299 -> 268; 4000,
    // 7^3: 129 -> 119, 207 -> 199, seven (one workgroup) 265 against 255 by now.  Even
    // numbers that way: from 4 % faster (eight, 7^3) to 19 % slower (two, 5^3); one
    // channel with helpers 39 -> 47.
    static constexpr bool kOneEach = E % 2 == 1 && E > 1 && kFit > 1;
    static constexpr int kY = kOneEach ? 8 : 4;
    static constexpr int kParts = kG / kY;
    static constexpr int kWorkers = E * kParts;                    // wavefronts that compute
    static constexpr int kThreads = 64 * (kOneEach ? (kWorkers + 3) / 4 * 4 : kWorkers);
    static constexpr int kOwnPieces = kM * E / 4;                  // of 16 bytes, a block's own rows
    static constexpr int kOwnEach = (kOwnPieces + kThreads - 1) / kThreads;   // per thread
    // the tile: kT * kT lines of eight cells along x, of 2 E pieces, and at either
    // end of a line kR cells, word by word
    static constexpr int kPieces = kT * kT * 2 * E;
    static constexpr int kPiecesEach = (kPieces + kThreads - 1) / kThreads;
    static constexpr int kEnds = 2 * kR * kT * kT * E;
    static constexpr int kEndsEach = (kEnds + kThreads - 1) / kThreads;
    static constexpr int kTaps = W * W;                           // of one dz
    // wavefronts per SIMD that the tile leaves room for.  No more than the
    // registers allow: 54 - 72 for windows of 3 and 71 - 80 for most of 5 are eight and
    // six, 104 - 120 for most of 7 are four.  (Five for 7: 4000 blocks of one channel 39.6 ->
    // 44.6 us, the others alike; three: alike.)  Five channels, 5^3, spill 3 registers with
    // six and gain all the same, five against six: 1000 blocks 26.6 -> 26.9 us, 12 000
    // 224 -> 208, 25 000 449 -> 417; four and six channels 153 -> 147 and 246 -> 221
    // at 12 000 without spilling, the others alike.
    // Windows of 3 whose workgroups are a wavefront per SIMD: six (40 000 blocks of
    // one to three channels with eight 44, 75, 130 us, with five to seven 44, 73 - 75, 108).
    static constexpr int kMostWaves = W == 3 ? (kThreads <= 256 ? 6 : 8) : (W == 5 ? 6 : 4);
    static constexpr int waves() {
        const int each = (kThreads / 64 + 3) / 4;   // of one workgroup
        const int fit = kFit < kMostWaves / each ? kFit : kMostWaves / each;
        return fit < 1 ? each : fit * each;
    }
};

struct ConvArgs {
    const float* in;
    const float* w;
    const int64_t* grid_indices;
    const int64_t* lut_g;   // [B, 27]
    float* out;
    const uint8_t* listed;  // [B]: rows of the others become zeros
    int64_t n_grids, B;
};

template <int E, int W>
__global__ __launch_bounds__((Shape<E, W>::kThreads), (Shape<E, W>::waves())) void
convolution_block8_kernel(ConvArgs a) {
    using S = Shape<E, W>;
    typedef float v4 __attribute__((ext_vector_type(4)));
    __shared__ __align__(16) float s_tile[S::kTileWords];
    __shared__ __align__(16) float s_out[S::kOutWords];
    __shared__ float s_w[S::kTapsHeld ? 1 : S::kWeightWords];
    __shared__ uint32_t s_nb[2][28];   // where the rows of the 27 neighbour blocks start, and the block's own
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = wave / S::kParts;             // the wavefront's channel
    const int y0 = wave % S::kParts * S::kY;     // and the first of its cells along y
    constexpr int R = S::kR, T = S::kT, kY = S::kY;

    // weights by channel and dz: one tap per lane, or all of the wavefront's channel
    float held[S::kTapsHeld ? W * W * W : 1];
    if constexpr (S::kTapsHeld) {
        const int ch = wave < S::kWorkers ? q : 0;
#pragma unroll
        for (int k = 0; k < W * W * W; ++k) {
            held[k] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(a.w[k * E + ch])));
        }
    } else {
        for (int t = tid; t < S::kWeightWords; t += S::kThreads) {
            const int tap = t & 63;
            const int dz = (t >> 6) % W;
            const int ch = (t >> 6) / W;
            s_w[t] = tap < S::kTaps ? a.w[(dz * S::kTaps + tap) * E + ch] : 0.f;
        }
    }
    // Along y or z: the block that tile coordinate `at` lies in (0, 1, 2: the block
    // before, the own, the next), and the cell there.
    auto block_at = [](int at) { return at < R ? 0 : (at >= R + kG ? 2 : 1); };
    auto cell_at = [](int at) { return (at - R + kG) % kG; };
    // This thread's pieces: neighbour << 14 | byte within that block's rows, and where
    // the four words go in the tile, two 16-bit places per register.
    uint32_t piece_src[S::kPiecesEach], piece_dst[S::kPiecesEach][2];
#pragma unroll
    for (int i = 0; i < S::kPiecesEach; ++i) {
        const int p = tid + i * S::kThreads < S::kPieces ? tid + i * S::kThreads : S::kPieces - 1;
        const int line = p / (2 * E), part = p - line * (2 * E);
        const int y = line % T, z = line / T;
        uint32_t place[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int e = 4 * part + c;
            const int cell = e / E;
            place[c] = static_cast<uint32_t>((e - cell * E) * S::kPlane + cell + R + T * y + S::kLayer * z);
        }
        piece_dst[i][0] = place[0] | (place[1] << 16);
        piece_dst[i][1] = place[2] | (place[3] << 16);
        const int nb = 1 + 3 * block_at(y) + 9 * block_at(z);
        piece_src[i] = (static_cast<uint32_t>(nb == 13 ? 27 : nb) << 14) |
                       static_cast<uint32_t>((kG * cell_at(y) + kG * kG * cell_at(z)) * E * 4 + 16 * part);
    }
    // and its words of the lines' ends: place in the tile << 17 | neighbour << 12 |
    // word within that block's rows
    uint32_t ends[S::kEndsEach];
#pragma unroll
    for (int i = 0; i < S::kEndsEach; ++i) {
        const int h = tid + i * S::kThreads < S::kEnds ? tid + i * S::kThreads : S::kEnds - 1;
        const int p = h / E, ch = h - p * E;
        const int line = p / (2 * R);
        const int y = line % T, z = line / T;
        int x = p % (2 * R);
        if (x >= R) x += kG;
        const int nb = block_at(x) + 3 * block_at(y) + 9 * block_at(z);
        const int cell = cell_at(x) + kG * cell_at(y) + kG * kG * cell_at(z);
        ends[i] = (static_cast<uint32_t>(ch * S::kPlane + x + T * y + S::kLayer * z) << 17) |
                  static_cast<uint32_t>(nb << 12) | static_cast<uint32_t>(cell * E + ch);
    }

    const TileWalk walk(a.n_grids);
    auto fetch_rows = [&](int64_t b) -> int32_t {   // lanes 0..26 neighbours, 27 the block
        if (tid > 27 || b >= walk.end) return -1;
        const int64_t g = a.grid_indices[b];
        if (g < 0 || g >= a.B) return -1;
        if (tid == 27) return static_cast<int32_t>(g);
        const int64_t row = a.lut_g[g * 27 + tid];
        return (row >= 0 && row < a.B) ? static_cast<int32_t>(row) : -1;
    };
    // Byte offsets fit 32 bits: the tensors are below 4 GiB, which the host checks, and
    // end at a multiple of 2048.  A missing block's rows are read beyond the tensor, where
    // the loads give zeros by themselves.
    constexpr uint32_t kBlockBytes = kM * E * 4, kMissing = 0xFFFFFFFFu, kBeyond = 0xFFFFFFF0u;
    auto start_of = [&](int32_t row) { return row < 0 ? kMissing : static_cast<uint32_t>(row) * kBlockBytes; };
    auto place_in = [&](uint32_t start, uint32_t byte) {
        return static_cast<int>(start == kMissing ? kBeyond : start + byte);
    };
    const auto in = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.in), 0,
                                                      static_cast<int>(static_cast<uint32_t>(a.B) * kBlockBytes),
                                                      0x00020000);
    v4 piece[S::kPiecesEach];
    float end[S::kEndsEach];
    auto load_block = [&](const uint32_t* nb) {
#pragma unroll
        for (int i = 0; i < S::kPiecesEach; ++i) {
            const int at = place_in(nb[piece_src[i] >> 14], piece_src[i] & 0x3FFFu);
            piece[i] = __builtin_bit_cast(v4, __builtin_amdgcn_raw_buffer_load_b128(in, at, 0, 0));
        }
#pragma unroll
        for (int i = 0; i < S::kEndsEach; ++i) {
            const int at = place_in(nb[(ends[i] >> 12) & 31u], (ends[i] & 0xFFFu) * 4u);
            end[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(in, at, 0, 0));
        }
    };

    int64_t blk = walk.next;
    int buf = 0;
    int32_t rows_reg = fetch_rows(blk);
    // Zeros for the blocks that are not listed: each workgroup looks at a share of
    // the flags, one per thread, while its first rows are on their way (a launch
    // of their own, one flag after the other per workgroup: 60 000 blocks, all
    // listed, 9.8 us).
    int32_t* const s_bare = reinterpret_cast<int32_t*>(s_out);
    static_assert(S::kOutWords > S::kThreads, "a row number per thread, and their number");
    for (int64_t first = blockIdx.x; first < a.B; first += static_cast<int64_t>(gridDim.x) * S::kThreads) {
        if (tid == 0) s_bare[S::kThreads] = 0;
        __syncthreads();
        const int64_t b = first + static_cast<int64_t>(gridDim.x) * tid;
        if (b < a.B && a.listed[b] == 0) {
            s_bare[atomicAdd(&s_bare[S::kThreads], 1)] = static_cast<int32_t>(b);
        }
        __syncthreads();
        const int bare = s_bare[S::kThreads];
        for (int j = 0; j < bare; ++j) {
            v4* rows = reinterpret_cast<v4*>(a.out) +
                       static_cast<uint64_t>(static_cast<uint32_t>(s_bare[j])) * (kM * E / 4);
            for (int f = tid; f < S::kOwnPieces; f += S::kThreads) {
                __builtin_nontemporal_store(v4{0.f, 0.f, 0.f, 0.f}, rows + f);
            }
        }
        __syncthreads();   // the list is written again by the next round
    }
    if (tid <= 27) s_nb[0][tid] = start_of(rows_reg);
    rows_reg = fetch_rows(blk + walk.step);
    __syncthreads();
    if (blk < walk.end) load_block(s_nb[0]);
    const int x = lane & 7, z = lane >> 3;
    const float* const window = s_tile + q * S::kPlane + x + T * y0 + S::kLayer * z;
    float* const result = s_out + (x + kG * y0) * E + z * S::kOutLayer + q;

    for (; blk < walk.end; blk += walk.step, buf ^= 1) {
        const uint32_t own = s_nb[buf][27];
#pragma unroll
        for (int i = 0; i < S::kPiecesEach; ++i) {
            if (S::kPieces % S::kThreads != 0 && tid + i * S::kThreads >= S::kPieces) continue;
#pragma unroll
            for (int c = 0; c < 4; ++c) s_tile[(piece_dst[i][c >> 1] >> (16 * (c & 1))) & 0xFFFFu] = piece[i][c];
        }
#pragma unroll
        for (int i = 0; i < S::kEndsEach; ++i) {
            if (S::kEnds % S::kThreads != 0 && tid + i * S::kThreads >= S::kEnds) continue;
            s_tile[ends[i] >> 17] = end[i];
        }
        if (tid <= 27) s_nb[buf ^ 1][tid] = start_of(rows_reg);
        __syncthreads();   // the tile is complete
        rows_reg = fetch_rows(blk + 2 * walk.step);
        if (blk + walk.step < walk.end) load_block(s_nb[buf ^ 1]);

        if (wave < S::kWorkers) {
            float acc[kY];
#pragma unroll
            for (int j = 0; j < kY; ++j) acc[j] = 0.f;
            // one layer of the window, tap(k) the k-th weight of it
            auto add_layer = [&](const float* layer, auto tap) {
#pragma unroll
                for (int y = 0; y < kY + 2 * R; ++y) {
                    float row[W];
#pragma unroll
                    for (int dx = 0; dx < W; ++dx) row[dx] = layer[T * y + dx];
#pragma unroll
                    for (int j = 0; j < kY; ++j) {
                        const int dy = y - j;
                        if (dy < 0 || dy >= W) continue;
#pragma unroll
                        for (int dx = 0; dx < W; ++dx) acc[j] = fmaf(row[dx], tap(dy * W + dx), acc[j]);
                    }
                }
            };
            if constexpr (S::kTapsHeld) {
#pragma unroll
                for (int dz = 0; dz < W; ++dz) {
                    add_layer(window + S::kLayer * dz, [&](int k) { return held[dz * S::kTaps + k]; });
                }
            } else {
#pragma unroll 1
                for (int dz = 0; dz < W; ++dz) {
                    const float taps = s_w[(q * W + dz) * 64 + lane];
                    add_layer(window + S::kLayer * dz, [&](int k) {
                        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(taps), k));
                    });
                }
            }
#pragma unroll
            for (int j = 0; j < kY; ++j) result[j * kG * E] = acc[j];
        }
        __syncthreads();   // the results are complete, and the tile has been read
        if (own != kMissing) {
            v4* rows = reinterpret_cast<v4*>(reinterpret_cast<char*>(a.out) + own);
#pragma unroll
            for (int i = 0; i < S::kOwnEach; ++i) {
                const int f = tid + i * S::kThreads;
                if (S::kOwnPieces % S::kThreads != 0 && f >= S::kOwnPieces) continue;
                const int out_z = f / (16 * E);
                __builtin_nontemporal_store(
                        *reinterpret_cast<const v4*>(s_out + 4 * f + (S::kOutLayer - 64 * E) * out_z), rows + f);
            }
        }
    }
}

// listed[b] = 1 for every block of the listing.
__global__ __launch_bounds__(kFillBlock) void mark_kernel(const int64_t* __restrict__ grid_indices,
                                                          int64_t n, int64_t B,
                                                          uint8_t* __restrict__ listed) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kFillBlock + threadIdx.x;
    if (i >= n) return;
    const int64_t g = grid_indices[i];
    if (g >= 0 && g < B) listed[g] = 1;
}

__global__ __launch_bounds__(kFillBlock) void clear_marks_kernel(uint8_t* __restrict__ listed, int64_t B) {
    const int64_t i = (static_cast<int64_t>(blockIdx.x) * kFillBlock + threadIdx.x) * 4;
    for (int64_t b = i; b < i + 4 && b < B; ++b) listed[b] = 0;
}

template <int E, int W>
int launch(const ConvArgs& a, hipStream_t s) {
    // as many workgroups as the device holds at once: they walk the listing, and
    // the flags of all blocks
    constexpr auto kernel = convolution_block8_kernel<E, W>;
    int64_t groups = static_cast<int64_t>(compute_units()) * resident_per_cu<kernel>(Shape<E, W>::kThreads);
    const int64_t most = a.n_grids > a.B ? a.n_grids : a.B;
    if (groups > most) groups = most;
    kernel<<<static_cast<unsigned>(groups), Shape<E, W>::kThreads, 0, s>>>(a);
    ASH_LAUNCH_CHECK();
    return 0;
}

template <int E>
int launch_window(const ConvArgs& a, int window, hipStream_t s) {
    switch (window) {
        case 3: return launch<E, 3>(a, s);
        case 5: return launch<E, 5>(a, s);
        default: return launch<E, 7>(a, s);
    }
}

}  // namespace
}  // namespace ash

using namespace ash;

extern "C" {

int ash_convolution_cube_supported(int64_t num_embeddings, int grid_dim, int window,
                                   int64_t embedding_dim, int32_t dtype) {
    return dtype == ASH_F32 && grid_dim == kG && (window == 3 || window == 5 || window == 7) &&
           embedding_dim >= 1 && embedding_dim <= kMaxChannels && num_embeddings >= 1 &&
           num_embeddings * embedding_dim * kM * 4 <= 0xFFFFFFFFll;
}

int ash_convolution_cube(const void* inputs, const void* weights, const int64_t* grid_indices,
                         const int64_t* lut_grid_nb2grid_idx, void* outputs, int64_t num_grids,
                         int64_t num_embeddings, int grid_dim, int window, int64_t embedding_dim,
                         int32_t dtype, uint8_t* listed, void* stream) {
    if (num_grids < 0 || num_embeddings < 1) ASH_FAIL("convolution_cube: bad sizes");
    if (!ash_convolution_cube_supported(num_embeddings, grid_dim, window, embedding_dim, dtype)) {
        ASH_FAIL("convolution_cube takes float32 blocks of 8^3 cells, windows of 3, 5 or 7, up to 8 "
                 "channels and up to 4 GiB");
    }
    if (inputs == nullptr || weights == nullptr || lut_grid_nb2grid_idx == nullptr ||
        outputs == nullptr || listed == nullptr || (num_grids > 0 && grid_indices == nullptr)) {
        ASH_FAIL("null pointer in convolution_cube");
    }
    if ((reinterpret_cast<uintptr_t>(inputs) | reinterpret_cast<uintptr_t>(outputs)) % 16 != 0) {
        ASH_FAIL("convolution_cube: inputs and outputs must be 16-byte aligned");
    }
    PointerGuard guard;
    ASH_HIP(guard.enter_for(inputs));
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t B = num_embeddings;
    clear_marks_kernel<<<static_cast<unsigned>((B + 4 * kFillBlock - 1) / (4 * kFillBlock)), kFillBlock, 0, s>>>(
            listed, B);
    ASH_LAUNCH_CHECK();
    if (num_grids > 0) {
        mark_kernel<<<static_cast<unsigned>((num_grids + kFillBlock - 1) / kFillBlock), kFillBlock, 0, s>>>(
                grid_indices, num_grids, B, listed);
        ASH_LAUNCH_CHECK();
    }
    const ConvArgs a = {static_cast<const float*>(inputs), static_cast<const float*>(weights),
                        grid_indices, lut_grid_nb2grid_idx, static_cast<float*>(outputs),
                        listed, num_grids, num_embeddings};
    switch (embedding_dim) {
        case 1: return launch_window<1>(a, window, s);
        case 2: return launch_window<2>(a, window, s);
        case 3: return launch_window<3>(a, window, s);
        case 4: return launch_window<4>(a, window, s);
        case 5: return launch_window<5>(a, window, s);
        case 6: return launch_window<6>(a, window, s);
        case 7: return launch_window<7>(a, window, s);
        default: return launch_window<8>(a, window, s);
    }
}

}  // extern "C"
