// How the workgroups of gemm_slim_kernel share its units.  constexpr, so that host and device (and a plain C++ compiler) see one rule.
#pragma once
#include <cstdint>

namespace tship {

// Units are (row tile, K chunk, column tile), column tile fastest; workgroup b of `grid` takes those from first(b) up to first(b + 1).
// A run is dealt out by weight, for a unit of the last K chunk, which may be short, costs less than the others.  Where there is a
// workgroup for every unit each takes one: by weight a workgroup could get the last unit of one chunk and the first of the next, loads
// the activations of both one after the other, and the kernel takes twice as long (whole calls on tiles of 16 columns, us, by weight / one
// each: Q8_0 18 x 64 x 9440 19.2 / 13.9, Q5_K 31 x 247 x 5376 18.2 / 13.8, Q4_K 26 x 799 x 16896 20.6 / 16.3).
struct UnitRuns {
    int row_tiles, k_chunks, n_tiles;
    int chunk_weight, last_weight;       // of a unit of all K chunks but the last, and of the last

    constexpr int first(int b, int grid) const
    {
        const int per_tile = k_chunks * n_tiles, units = row_tiles * per_tile;
        if (units <= grid) return b < units ? b : units;
        const int64_t front = (int64_t)(k_chunks - 1) * n_tiles * chunk_weight, weight = front + (int64_t)n_tiles * last_weight;
        const int64_t at = row_tiles * weight * b / grid;
        const int tile = (int)(at / weight), rest = (int)(at - tile * weight);
        return tile * per_tile + (rest < front ? rest / chunk_weight : (k_chunks - 1) * n_tiles + (rest - (int)front) / last_weight);
    }
};

}  // namespace tship
