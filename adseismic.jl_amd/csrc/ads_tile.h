// ads_tile.h -- what the register-tile kernels of the acoustic and the elastic scheme share: lane
// moves, wave-uniform values and the cutting of a grid's axis into tiles with a halo.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

#include "ads_common.h"

namespace ads {

// lane L receives lane L + 1's (L - 1's) value; the last (first) lane receives 0
template <int CTRL> __device__ inline float tile_dpp(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL> __device__ inline double tile_dpp(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
template <typename T> __device__ inline T lane_east(T v) { return tile_dpp<0x130>(v); }
template <typename T> __device__ inline T lane_west(T v) { return tile_dpp<0x138>(v); }
// a value that every lane holds alike, as a scalar
__device__ inline float uniform(float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); }
__device__ inline double uniform(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// Makes a value opaque here, so that what follows from it is computed where it is used instead of
// being kept in registers for every row across the levels.
__device__ inline void recompute(float &v) { asm volatile("" : "+v"(v)); }
__device__ inline void recompute(double &v) { asm volatile("" : "+v"(v)); }

// Rows r with lo <= r0 + r < hi (wave-uniform).
template <int R> __device__ inline uint32_t row_mask(int r0, int lo, int hi)
{
    const int a = min(max(lo - r0, 0), R), b = min(max(hi - r0, 0), R);
    return __builtin_amdgcn_readfirstlane((1u << b) - (1u << min(a, b)));
}

// Cuts [lo, hi) into equal pieces whose extents (halo H, clipped to [0, n)) fit in cap cells.
static inline std::vector<int> tile_cuts(int lo, int hi, int H, int n, int cap)
{
    // pieces away from the grid's edges hold at most cap - 2 H cells, the two at its edges H more
    const int len = hi - lo, in = std::max(cap - 2 * H, 1);
    for (int k = std::max(1, (len - 2 * H) / in);; k++) {
        std::vector<int> c;
        const int size = (len + k - 1) / k;
        for (int x = lo; x < hi; x += size) c.push_back(x);
        c.push_back(hi);
        bool ok = true;
        for (size_t q = 0; q + 1 < c.size(); q++)
            ok = ok && std::min(c[q + 1] + H, n) - std::max(c[q] - H, 0) <= cap;
        if (ok || size <= 1) return c;
    }
}

}  // namespace ads
