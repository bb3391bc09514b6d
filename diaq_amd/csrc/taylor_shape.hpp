// Launch shapes of taylor_rows_kernel (expm_dense.hip) and the room that its norms take. Host arithmetic alone, without
// HIP, so that its bounds can be checked without a GPU.
#pragma once

#include <cstdint>

namespace dq {

constexpr int TAYLOR_BATCH = 32;       // terms of a launch that writes norms
constexpr int64_t TAYLOR_MAX_N = 8192;  // rows of the largest shape

struct TaylorShape {
    int threads, cols, rows;  // lanes of a workgroup, columns per lane, rows of a workgroup
};

// A row per workgroup while that fills the chip, then as many as 128 KB of LDS hold. shape: an index into this list.
constexpr TaylorShape TAYLOR_SHAPES[] = {{256, 1, 1}, {512, 1, 2}, {1024, 1, 4}, {1024, 2, 4}, {1024, 4, 2}, {1024, 8, 1}};

inline int taylor_shape(int64_t N) {
    int i = 0;
    while (i < 5 && static_cast<int64_t>(TAYLOR_SHAPES[i].threads) * TAYLOR_SHAPES[i].cols < N) ++i;
    return i;
}

inline int64_t taylor_grid(int64_t N) {
    const int rows = TAYLOR_SHAPES[taylor_shape(N)].rows;
    return (N + rows - 1) / rows;
}

// The doubles that a launch of `terms` terms writes as shares of the norms, and those that there is room for.
inline int64_t taylor_parts(int64_t N, int terms, bool norms) { return norms ? terms * taylor_grid(N) : 0; }
inline int64_t taylor_parts_room(int64_t N) { return TAYLOR_BATCH * taylor_grid(N); }

}  // namespace dq
