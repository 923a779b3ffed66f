// How persistent workgroups share a run of tiles between the XCDs.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ash {

constexpr int kXcds = 8;

// Tile walk: workgroup w serves XCD (w mod 8); each XCD owns a contiguous
// eighth of the tiles and its workgroups stride through it.
struct TileWalk {
    int64_t next;
    int64_t end;
    int64_t step;
    __device__ __forceinline__ TileWalk(int64_t ntiles) {
        const int64_t per_xcd = (ntiles + kXcds - 1) / kXcds;
        const int xcd = blockIdx.x % kXcds;
        const int slot = blockIdx.x / kXcds;
        step = (gridDim.x + kXcds - 1 - xcd) / kXcds;  // workgroups on this XCD
        next = xcd * per_xcd + slot;
        end = (xcd + 1) * per_xcd;
        if (end > ntiles) end = ntiles;
        if (step < 1) step = 1;
    }
};

}  // namespace ash
