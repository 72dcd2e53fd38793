// The cut of a batch's columns into ranges (lbman3d_amd/csrc/batch_split.hpp):
// no GPU. Every plane of every column is in one piece, pieces keep to the
// chunk length, ranges to the number of blocks, and none costs much more than
// its share; a set whose cost does not fit 32 bits is cut like any other.
#include <cstdio>
#include <cstdlib>

#include "../../lbman3d_amd/csrc/batch_split.hpp"

using namespace lbm;

namespace {
int g_failures = 0;
void expect(bool ok, const char* what, const char* where) {
    if (ok) return;
    ++g_failures;
    std::printf("FAILED: %s (%s)\n", what, where);
}

void check(const std::vector<BatchColumns>& sims, int zc, int slots, const char* where) {
    const BatchSplit s = split_columns(sims, zc, slots);
    expect(s.ranges() >= 1 && s.ranges() <= slots, "ranges", where);
    expect(s.first.front() == 0 && s.first.back() == (int)s.items.size(), "range ends", where);
    size_t at = 0;
    long total = 0, planes = 0;
    for (const BatchColumns& c : sims)
        for (int txy = 0; txy < c.columns; ++txy)
            for (int z = 0; z < c.nz; ++at) {
                if (at >= s.items.size()) return expect(false, "planes missing", where);
                const BatchItem& it = s.items[at];
                if (it.sim != c.sim || it.txy != txy || it.z0 != z || it.z1 <= z || it.z1 > c.nz || it.z1 - z > zc)
                    return expect(false, "piece", where);
                total += kPieceStart + (it.z1 - z) * (c.walls ? kWallPlane : kPlane);
                planes += it.z1 - z;
                z = it.z1;
            }
    expect(at == s.items.size(), "pieces", where);
    long worst = 0;
    at = 0;
    for (int r = 0; r < s.ranges(); ++r) {
        expect(s.first[r] < s.first[r + 1], "empty range", where);
        long load = 0;
        for (int i = s.first[r]; i < s.first[r + 1]; ++i) {
            bool walls = false;
            for (const BatchColumns& c : sims)
                if (c.sim == s.items[i].sim) walls = c.walls;
            load += kPieceStart + (s.items[i].z1 - s.items[i].z0) * (walls ? kWallPlane : kPlane);
        }
        worst = std::max(worst, load);
    }
    // The share, the start and shortest piece that end a range early, and the
    // plane that joins its last piece.
    expect(worst <= total / slots + 2 * (kPieceStart + (kPieceMin + 1) * kWallPlane) + total / (slots * 4), "costliest range", where);
}
}  // namespace

int main() {
    std::srand(5);
    for (int k = 0; k < 200; ++k) {
        std::vector<BatchColumns> sims;
        const int n = 1 + std::rand() % 40;
        for (int i = 0; i < n; ++i) sims.push_back({i, 1 + std::rand() % 24, 1 + std::rand() % 100, std::rand() % 2 == 0});
        const int slots[] = {1, 2, 7, 200, 512, 100000};
        const int zc[] = {8, 16, 32, 64};
        char where[64];
        std::snprintf(where, sizeof where, "mix %d", k);
        check(sims, zc[std::rand() % 4], slots[std::rand() % 6], where);
    }
    check({{0, 1, 1, true}}, 64, 512, "one plane");
    // four columns of one cell's width, 286 million planes, on one block
    check({{0, 1, 71500000, false}, {1, 1, 71500000, true}, {2, 1, 71500000, true}, {3, 1, 71500000, true}}, 64, 1, "long");
    if (!g_failures) std::printf("ok\n");
    return g_failures ? 1 : 0;
}
