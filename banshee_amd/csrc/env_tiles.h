// Tiling of an environment map for its projection. Plain C++ when compiled on the host (also by the host
// tests).
#pragma once

#include <algorithm>
#include <cstdint>

#if defined(__HIPCC__)
#define BSH_ENV_HD __host__ __device__ inline
#else
#define BSH_ENV_HD inline
#endif

namespace bsh {

constexpr int kShBlock = 256, kShTile = 256;
// Blocks of the environment projection: two per CU.
constexpr int kEnvMaxBlocks = 512;

// `cols` columns and `rows` rows per block, nx x ny blocks, about two per CU where the map is large
// enough and at most kEnvMaxBlocks, or more where rows per block are at their limit.
struct EnvTiles
{
    int cols, rows, nx, ny;
};
inline EnvTiles env_tiles(int W, int H)
{
    EnvTiles t;
    t.cols = 1;
    while (t.cols < W && t.cols < kShTile) t.cols *= 2;
    t.nx = (int)(((int64_t)W + t.cols - 1) / t.cols);
    const int sub = kShBlock / t.cols;   // rows a block reads at a time
    const int want = std::max(1, kEnvMaxBlocks / t.nx);
    t.rows = std::max(sub, (int)(((int64_t)H + want - 1) / want));
    t.rows = std::min(t.rows, kShBlock);   // a block's angle table
    t.ny = (int)(((int64_t)H + t.rows - 1) / t.rows);
    return t;
}

// A block's first column and its rows [row0, row1).
struct EnvTile
{
    int col0, row0, row1;
};
BSH_ENV_HD EnvTile env_tile(uint32_t block, EnvTiles t, int H)
{
    const int by = (int)(block / (uint32_t)t.nx), row0 = by * t.rows;
    return EnvTile{(int)(block % (uint32_t)t.nx) * t.cols, row0, H - row0 < t.rows ? H : row0 + t.rows};
}

}  // namespace bsh
