// Device types and launch helpers shared by the HIP sources.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace hgm {

template <class T> struct Vec;
template <> struct Vec<double> { using type = double2; };
template <> struct Vec<float> { using type = float2; };

template <class V, class T>
__device__ __forceinline__ V cmul(T mr, T mi, V a) {
    V o;
    o.x = mr * a.x - mi * a.y;
    o.y = mr * a.y + mi * a.x;
    return o;
}

template <class V, class T>
__device__ __forceinline__ V cmul2(T ar, T ai, V x, T br, T bi, V y) {
    V o;
    o.x = ar * x.x - ai * x.y + br * y.x - bi * y.y;
    o.y = ar * x.y + ai * x.x + br * y.y + bi * y.x;
    return o;
}

inline uint64_t max_blocks(int block) { return 0xffffffffull / (uint64_t)block; }

inline int64_t tile_grid(int64_t n_tiles, int block) {
    int64_t g = n_tiles < (int64_t(1) << 22) ? n_tiles : (int64_t(1) << 22);
    if ((uint64_t)g > max_blocks(block)) g = (int64_t)max_blocks(block);
    return g;
}

}  // namespace hgm
