// How persistent workgroups share a run of tiles between the XCDs.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

namespace ash {

constexpr int kXcds = 8;

// Tile walk: workgroup w serves XCD (w mod 8); each XCD owns a contiguous
// eighth of the tiles and its workgroups stride through it.
struct TileWalk {
    int64_t next;
    int64_t end;
    int64_t step;
    __device__ __forceinline__ TileWalk(int64_t ntiles) : TileWalk(ntiles, blockIdx.x, gridDim.x) {}
    // the `group`-th of `groups` workgroups, on the XCD of its number
    __device__ __forceinline__ TileWalk(int64_t ntiles, unsigned group, unsigned groups) {
        const int64_t per_xcd = (ntiles + kXcds - 1) / kXcds;
        const int xcd = group % kXcds;
        const int slot = group / kXcds;
        step = (groups + kXcds - 1 - xcd) / kXcds;  // workgroups on this XCD
        next = xcd * per_xcd + slot;
        end = (xcd + 1) * per_xcd;
        if (end > ntiles) end = ntiles;
        if (step < 1) step = 1;
    }
};

// What does not change for a device of the process, asked once for each (0: not
// yet; threads that ask at the same time get the same answer).
class PerDevice {
  public:
    template <typename Ask>
    int get(const Ask& ask, int otherwise) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return otherwise;
        const bool kept = dev >= 0 && dev < kDevices;
        int n = kept ? known_[dev].load(std::memory_order_relaxed) : 0;
        if (n > 0) return n;
        if (ask(dev, &n) != hipSuccess || n < 1) {
            (void)hipGetLastError();
            return otherwise;
        }
        if (kept) known_[dev].store(n, std::memory_order_relaxed);
        return n;
    }

  private:
    static constexpr int kDevices = 16;
    std::atomic<int> known_[kDevices] = {};
};

inline int compute_units() {
    static PerDevice units;
    return units.get([](int dev, int* n) {
        return hipDeviceGetAttribute(n, hipDeviceAttributeMultiprocessorCount, dev); }, 256);
}

// Workgroups of `Kernel` that a CU holds at once as far as registers, wavefronts
// and static LDS go.
template <auto Kernel>
int resident_per_cu(int threads) {
    static PerDevice resident;
    return resident.get([threads](int, int* n) {
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(n, Kernel, threads, 0); }, 1);
}

}  // namespace ash
