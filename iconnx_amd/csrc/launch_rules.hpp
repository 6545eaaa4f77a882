// Launch rules that are plain arithmetic: no HIP header, so that a host program (a test on the
// CPU) can walk them over sizes that no test would allocate.
#pragma once

#include <algorithm>
#include <cstdint>

namespace icx {

constexpr uint32_t kChainThreads = 256;  // lanes of a chain_any_kernel block
constexpr uint32_t chain_in_flight(int vec) { return vec == 4 ? 2 : 8; }  // chunks of a lane per step

// chain_any_kernel over `chunks` chunks (of `vec` floats) of rows of C chunks.  lane_cols: every
// chunk of a lane has the same columns, because a lane takes one chunk or the grid stride is a
// multiple of the row (of `unit` blocks, lcm(256, C) lanes), so that column factors are fetched
// once a lane.  That takes one round of the chip's resident blocks (up to 2048 of them), or
// three chunks a lane (two of four floats), to pay; other wide rows fetch column factors per
// chunk, a lane taking a whole step of chunks.  Whole rows / per chunk, in us, a column chain:
// 1000 x 1025 5.2 / 5.8, 1200 x 8191 21.7 / 23.2, 2000 x 16383 45 / 67, 700 x 12004 with a
// full-tensor Add 17.5 / 18.7; past the line 300 x 2049 7.4 / 5.5, 300 x 8191 18.5 / 10.1,
// 1 x 300001 139 / 5.3, 1 x 1000003 684 / 5.7, 3 x 5000004 2140 / 38.
// The grid is at most 16384 blocks, so that the 32-bit chunk index (chunks < 2^31) plus a step of
// at most 8 x 16384 x 256 = 2^25 cannot wrap.
struct ChainGrid {
    uint32_t blocks;
    bool lane_cols;
};
inline ChainGrid chain_grid(uint64_t chunks, uint64_t C, int vec) {
    const uint64_t one = (chunks + kChainThreads - 1) / kChainThreads;  // one chunk a lane
    if (one <= 1024) return {(uint32_t)one, true};
    uint64_t a = kChainThreads, b = C;
    while (b) {
        const uint64_t r = a % b;
        a = b;
        b = r;
    }
    const uint64_t unit = C / a;
    if (unit <= 1024) return {(uint32_t)(1024 / unit * unit), true};
    if (unit <= 2048) return {(uint32_t)std::min(unit, one), true};
    if (unit <= 16384 && (vec == 4 ? 2 : 3) * unit <= one) return {(uint32_t)unit, true};
    const uint64_t u = chain_in_flight(vec);
    return {(uint32_t)std::min<uint64_t>((one + u - 1) / u, 1024), false};
}

// Rows a block of layer_norm_kernel takes, or 0 where layer_norm_wide_kernel (32 rows a block)
// runs: blocks of 4096 floats, in fewer rows where that leaves the chip under two blocks per CU;
// rows too wide for LDS, and more blocks than a launch holds (HIP's limit is 2^32 - 1 threads: one
// row a block passes it at 2^24 rows), go to the wide kernel.
constexpr uint64_t kLnThreads = 256;
constexpr uint64_t kLnMaxCols = 12288;  // one staged row: 48 KB of LDS
inline int layer_norm_rows(uint64_t rows, uint64_t cols, uint64_t cus) {
    if (cols > kLnMaxCols) return 0;
    const auto blocks = [&](uint64_t rpb) { return (rows + rpb - 1) / rpb; };
    uint64_t rpb = 32;
    while (rpb > 1 && rpb * cols > 4096) rpb /= 2;
    while (rpb > 1 && blocks(rpb) < 2 * cus) rpb /= 2;
    return blocks(rpb) * kLnThreads > 0xffffffffull ? 0 : (int)rpb;
}

}  // namespace icx
