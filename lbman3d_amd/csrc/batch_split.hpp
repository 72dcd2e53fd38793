// batch_split.hpp — the cut of a batch's columns into one range of work per
// block of the third-pipeline kernel (host code, no HIP).
#pragma once

#include <algorithm>
#include <vector>

namespace lbm {

// Work item of the third-pipeline kernel: planes [z0, z1) of column tile txy
// (= tx + ty * ntx) of simulation sim.
struct BatchItem {
    int sim, txy, z0, z1;
};

// The column tiles of one simulation.
struct BatchColumns {
    int sim, columns, nz;
    bool walls;   // runs the wall-aware form
};

struct BatchSplit {
    std::vector<BatchItem> items;
    std::vector<int> first;   // first item of each range, and the number of items
    int ranges() const { return (int)first.size() - 1; }
};

// Costs, in eighths of a periodic plane: a piece of n planes also fills the
// pipeline, about two planes' time, and the wall-aware form takes about an
// eighth more per plane. 64 bits: a range may hold everything.
constexpr long kPlane = 8, kWallPlane = 9;
constexpr long kPieceStart = 2 * kPlane;
constexpr int kPieceMin = 4;   // planes; 6 boxes: 2 the same, 8: 45 -> 57 us

// Greedy cut with every range's cost at most `bound` (or one piece), pieces of
// at most zc planes.
inline void cut_columns(const std::vector<BatchColumns>& sims, int zc, long bound, BatchSplit& out) {
    out.items.clear();
    out.first.assign(1, 0);
    long load = 0;
    for (const BatchColumns& s : sims) {
        const long wp = s.walls ? kWallPlane : kPlane;
        for (int txy = 0; txy < s.columns; ++txy)
            for (int z = 0; z < s.nz;) {
                const int left = s.nz - z;
                const long room = (bound - load - kPieceStart) / wp;
                if (room < std::min(kPieceMin, left) && load > 0) {
                    out.first.push_back((int)out.items.size());
                    load = 0;
                    continue;
                }
                int n = (int)std::min<long>(std::min(left, zc), std::max<long>(room, kPieceMin));
                if (left - n == 1 && left <= zc) n = left;   // one plane more, not a piece of one
                out.items.push_back({s.sim, txy, z, z + n});
                load += kPieceStart + n * wp;
                z += n;
            }
    }
    out.first.push_back((int)out.items.size());
}

// The columns, one after another, in at most `slots` ranges whose costliest is
// the cheapest possible (by bisection over its cost).
inline BatchSplit split_columns(const std::vector<BatchColumns>& sims, int zc, int slots) {
    BatchSplit split;
    long lo = kPieceStart + kPlane * kPieceMin, hi = lo;
    auto fits = [&](long bound) {
        cut_columns(sims, zc, bound, split);
        return split.ranges() <= slots;
    };
    while (!fits(hi)) hi *= 2;
    while (lo < hi) {
        const long mid = (lo + hi) / 2;
        if (fits(mid)) hi = mid;
        else lo = mid + 1;
    }
    cut_columns(sims, zc, hi, split);
    return split;
}

}  // namespace lbm
