// Near-field source staging of the 3D direct kernel (256 threads; in 2D, with at
// most 13 boxes to a list, a stage per box is the faster: 38 against 46 us on
// 10^5 mixture points): the sources of a unit's source boxes lie in many short ranges (a
// leaf holds a few to 100), so up to 64 ranges are scanned at once and their
// sources staged 256 at a time, whichever boxes they come from -- two dependent
// loads and two barriers per 256 sources instead of per box.  Every wavefront
// scans the ranges for itself: no barrier, and a unit of one box pays nothing.
#pragma once

#include "fgtpw_impl.hpp"

namespace fgtpw {

constexpr int NEAR_RANGES = 64;
struct NearBatch {          // a wavefront's own copy
    int off[NEAR_RANGES];   // first staged position of every range
    int st[NEAR_RANGES];    // its first source
};

// ranges list[b0 .. b0 + n), n <= NEAR_RANGES; returns the number of their
// sources
__device__ __forceinline__ int near_ranges(NearBatch& B, const int* list, const int2* se, int b0,
                                           int n)
{
    const int lane = threadIdx.x & 63;
    int c = 0, s = 0;
    if (lane < n) {
        const int2 r = se[list[b0 + lane]];
        s = r.x;
        c = max(r.y - r.x, 0);
    }
    int x = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    // a wavefront's LDS accesses keep their order; the fences hold the compiler
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    B.off[lane] = x - c;
    B.st[lane] = s;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    return __shfl(x, 63);
}

// the source at staged position p of a batch of n ranges
__device__ __forceinline__ int near_source(const NearBatch& B, int n, int p)
{
    int lo = 0, hi = n - 1;  // the last range that starts at or before p
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (B.off[mid] <= p) lo = mid; else hi = mid - 1;
    }
    return B.st[lo] + p - B.off[lo];
}

// threads per target (neighbouring lanes, a power of two, at most 64) when
// 256 threads take cnt <= 256 targets
__device__ __forceinline__ int near_split(int cnt)
{
    int k = 1;
    while (k < 64 && 2 * k * cnt <= 256) k *= 2;
    return k;
}

}  // namespace fgtpw
