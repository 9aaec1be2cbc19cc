// Bin and sort keys of list elements, shared by the bin sorts.
#pragma once

#include "fgx_internal.h"

namespace fgx {

__device__ __forceinline__ uint32_t load_count(const uint32_t* d_n, uint32_t n_cap) {
    if (!d_n) return n_cap;
    const uint32_t n = __hip_atomic_load(d_n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return n < n_cap ? n : n_cap;
}

// ================================================================ bin keys
struct KeyArgs {
    int32_t mode;        // 0: message bin (clamped, MessageSpatial3DDevice.cuh:646-672)
                         // 1: agent sort key (unclamped, CUDASimulation.cu:372-408)
                         // 2: bucket key, x holds int32 keys (MessageBucket.cu:58-72)
    int32_t dims;
    float min[3];
    float radius;
    float width[3];
    uint32_t grid[3];
    uint32_t key_mask;   // mode 1: (1 << key_bits) - 1
    int32_t key_min;     // mode 2: lowest key
    uint32_t keys;       // mode 2: number of keys
};

__device__ __forceinline__ uint32_t bin_key(const KeyArgs& k, float x, float y, float z) {
    if (k.mode == 2) {
        // keys outside the range were reported by setKey; clamp so they stay in the table
        const int v = __float_as_int(x) - k.key_min;
        return v < 0 ? 0u : ((uint32_t)v >= k.keys ? k.keys - 1u : (uint32_t)v);
    }
    if (k.mode == 0) {
        int c[3];
        const float p[3] = {x, y, z};
        for (int a = 0; a < 3; ++a) {
            if (a < k.dims) {
                const int g = (int)floorf((p[a] - k.min[a]) / k.radius);
                const int hi = (int)k.grid[a] - 1;
                c[a] = g < 0 ? 0 : (g > hi ? hi : g);
            } else {
                c[a] = 0;
            }
        }
        return (uint32_t)c[2] * k.grid[0] * k.grid[1] + (uint32_t)c[1] * k.grid[0] + (uint32_t)c[0];
    } else {
        const int gx = (int)floorf(((x - k.min[0]) / k.width[0]) * (float)k.grid[0]);
        const int gy = (int)floorf(((y - k.min[1]) / k.width[1]) * (float)k.grid[1]);
        uint32_t b;
        if (k.dims == 3) {
            const int gz = (int)floorf(((z - k.min[2]) / k.width[2]) * (float)k.grid[2]);
            b = (uint32_t)gz * k.grid[0] * k.grid[1] + (uint32_t)gy * k.grid[0] + (uint32_t)gx;
        } else {
            b = (uint32_t)gy * k.grid[0] + (uint32_t)gx;
        }
        return b & k.key_mask;
    }
}

}  // namespace fgx
