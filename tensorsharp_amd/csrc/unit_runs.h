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

    // What the run that takes longest costs: per_kt for each k-tile of a wavefront (`full` in a unit, `last` in those of the last K chunk),
    // per_unit for each unit, per_cross for each further row tile or K chunk that the run enters.  Looked at are the runs inside one chunk
    // and those across its edges (twelve of them, evenly spread, where there are more).
    constexpr int64_t longest(int grid, int full, int last, int per_kt, int per_unit, int per_cross) const
    {
        const int64_t whole = (int64_t)full * per_kt + per_unit, end = (int64_t)last * per_kt + per_unit;
        const int segments = row_tiles * k_chunks, edges = segments - 1;
        if ((int64_t)segments * n_tiles <= grid) return k_chunks > 1 ? whole : end;
        const int64_t weight = (int64_t)n_tiles * ((int64_t)(k_chunks - 1) * chunk_weight + last_weight), total = row_tiles * weight;
        const int64_t n_end = (total + (int64_t)grid * last_weight - 1) / ((int64_t)grid * last_weight);
        int64_t worst = end * (n_end < n_tiles ? n_end : n_tiles);
        if (k_chunks > 1) {
            const int64_t n = (total + (int64_t)grid * chunk_weight - 1) / ((int64_t)grid * chunk_weight), cost = whole * (n < n_tiles ? n : n_tiles);
            if (cost > worst) worst = cost;
        }
        for (int i = 0; i < (edges < 12 ? edges : 12); ++i) {
            const int s = 1 + (edges <= 12 ? i : (int)((int64_t)i * edges / 12));            // the edge in front of segment s
            const int64_t before = (s / k_chunks * weight + (int64_t)(s % k_chunks) * n_tiles * chunk_weight) * grid;
            if (before % total == 0) continue;                                                // (a run begins there)
            const int b = (int)(before / total), lo = first(b, grid), hi = first(b + 1, grid);
            int64_t cost = -(int64_t)per_cross;
            for (int u = lo, next = lo; u < hi; u = next) {
                const int segment = u / n_tiles;
                next = (segment + 1) * n_tiles < hi ? (segment + 1) * n_tiles : hi;
                cost += (next - u) * (segment % k_chunks == k_chunks - 1 ? end : whole) + per_cross;
            }
            if (cost > worst) worst = cost;
        }
        return worst;
    }
};

}  // namespace tship
