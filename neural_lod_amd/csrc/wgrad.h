// How the weight gradients dW_l = sum_q delta_l[u][q] input_l[k][q] of one
// network are split over workgroups: 64 x 64 tiles of every matrix (grid.y)
// times chunks of queries (grid.x).  A wave keeps a whole tile (4 x 4 MFMA
// tiles, 64 accumulators a lane), so an operand fragment feeds four MFMAs, and
// the block's four waves take every fourth step of the chunk; they add up
// through LDS and write one partial matrix per chunk.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "nlod_common.h"

namespace nlod {

constexpr uint32_t kWgradTile = 64;

struct WgradItem {
    uint32_t layer, row0, col0;  // matrix 0 .. L and the tile's first row and column
};

// Matrices: the input one [W][cols0], L - 1 hidden ones [W][W], the output one [out_rows][W].
struct WgradShape {
    uint32_t W, cols0, L, out_rows;
};

__host__ __device__ inline uint32_t wgrad_blocks(uint32_t n) { return (n + kWgradTile - 1) / kWgradTile; }

inline uint32_t wgrad_items(const WgradShape& s) {
    const uint32_t rb = wgrad_blocks(s.W);
    return rb * wgrad_blocks(s.cols0) + (s.L - 1) * rb * rb + wgrad_blocks(s.out_rows) * rb;
}

__device__ inline WgradItem wgrad_item(uint32_t item, const WgradShape& s) {
    const uint32_t rb = wgrad_blocks(s.W), cb0 = wgrad_blocks(s.cols0);
    if (item < rb * cb0) return {0, item / cb0 * kWgradTile, item % cb0 * kWgradTile};
    item -= rb * cb0;
    if (item < (s.L - 1) * rb * rb)
        return {1 + item / (rb * rb), item % (rb * rb) / rb * kWgradTile, item % rb * kWgradTile};
    item -= (s.L - 1) * rb * rb;
    return {s.L, item / rb * kWgradTile, item % rb * kWgradTile};
}

// Chunks of `steps` steps: four blocks per CU over all tiles, as long as a
// wave still gets two steps (fewer chunks also mean fewer partials to add).
inline uint32_t wgrad_chunks(uint32_t items, uint32_t steps) {
    const uint32_t fill = std::max<uint32_t>(1, 4 * (uint32_t)cu_count() / items);
    return std::max<uint32_t>(1, std::min(fill, div_round_up(steps, 8)));
}

// Adds the accumulators of a block's four waves into wave 0's, waves 1 .. 3 in
// a fixed order.  lds: 2 x TILES x 64 float4.
template <int TILES, typename Acc>
__device__ __forceinline__ void wgrad_add_waves(Acc (&acc)[TILES], float4* lds) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto put = [&](int slot) {
#pragma unroll
        for (int t = 0; t < TILES; ++t)
            lds[(slot * TILES + t) * 64 + lane] = {acc[t][0], acc[t][1], acc[t][2], acc[t][3]};
    };
    auto add = [&](int slot) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const float4 v = lds[(slot * TILES + t) * 64 + lane];
            acc[t][0] += v.x;
            acc[t][1] += v.y;
            acc[t][2] += v.z;
            acc[t][3] += v.w;
        }
    };
    if (wave >= 2) put(wave - 2);
    __syncthreads();
    if (wave < 2) add(wave);
    __syncthreads();
    if (wave == 1) put(0);
    __syncthreads();
    if (wave == 0) add(0);
}

}  // namespace nlod
