// Host check of hm_tiles.hpp: the kernels' own tile shapes and thread placement.
// - small_div is the exact quotient for every pair up to 512;
// - over extents along the axis and rows of columns across it, the tiles of the
//   fused multi-species flux (large and small) and of the diffusive flux visit
//   every midpoint face or cell at least once and write every output face once;
// - the cells, sensor cells and faces of a small tile have one thread and one
//   LDS slot each (the shapes' bounds are asserted where they are defined).
// Prints the first failure and exits 1.
#include <cstdio>
#include <vector>

#include "../hamers_amd/csrc/hm_tiles.hpp"

using namespace hm;

struct Kind {
    const char* name;
    int threads, shared, dim;
    bool small, diff;
};

static int check(const Kind& t, int axis, int nA, int nU, int nV) {
    int R = 0, W = 0, ntA = 0;
    if (t.diff)
        dtile_shape(t.dim, nA, R, W, ntA);
    else
        mtile_shape(nA, R, W, ntA, t.small, t.dim);
    if (R * W > t.threads || W < 1) return 1;
    const uint32_t mul = small_div_mul(uint32_t(axis == 0 ? R : W));
    std::vector<int> in(size_t(nU) * nV * (nA + 1 + t.shared), 0), out(size_t(nU) * nV * (nA + 1), 0);
    const int columns = nU * nV, tiles = ntA * ((columns + W - 1) / W);
    for (int tile = 0; tile < tiles; tile++) {
        const int tw = tile / ntA, tA = tile % ntA;
        for (int lane = 0; lane < t.threads; lane++) {
            uint32_t r, w, u, v;
            tile_place(axis, uint32_t(lane), uint32_t(R), uint32_t(W), mul, r, w);
            tile_column(uint32_t(tw) * uint32_t(W), w, uint32_t(W), uint32_t(nU), u, v);
            const int at = tA * (R - t.shared) + int(r);  // midpoint face, or cell + 6
            if (lane >= R * W || at >= nA + 1 + t.shared || v >= uint32_t(nV)) continue;
            const size_t col = size_t(v) * nU + u;
            if (u >= uint32_t(nU)) return 1;
            in[col * (nA + 1 + t.shared) + at]++;
            // a face needs the neighbouring midpoint faces of its own, or three nodes below and two above
            const int below = t.diff ? 6 : 1, above = t.diff ? 5 : 1, face = at - below;
            if (int(r) < below || int(r) > R - 1 - above || face > nA) continue;
            if (face < 0) return 1;
            out[col * (nA + 1) + face]++;
        }
    }
    for (int x : in)
        if (x < 1) return 1;
    for (int x : out)
        if (x != 1) return 1;
    return 0;
}

int main() {
    for (uint32_t d = 1; d <= 512; d++)
        for (uint32_t x = 0; x <= 512; x++)
            if (small_div(x, small_div_mul(d)) != x / d) {
                std::printf("small_div %u / %u\n", x, d);
                return 1;
            }
    for (int dim = 1; dim <= 3; dim++)
        for (int nA = 1; nA < 2000; nA++) {
            int R = 0, W = 0, ntA = 0;
            mtile_shape(nA, R, W, ntA, true, dim);
            const int cells = (R + 5) * W, sensor = (R + 1) * W;
            if (R * W > kSmallThreads || cells > kSmallCells || sensor > kSmallSensor ||
                int(small_sensor_first(uint32_t(cells))) < cells ||
                int(small_sensor_first(uint32_t(cells))) + sensor > kMTileThreads) {
                std::printf("small tile of %d cells, %dD\n", nA, dim);
                return 1;
            }
        }
    const Kind kinds[] = {{"flux", kMTileThreads, 2, 3, false, false}, {"small", kSmallThreads, 2, 3, true, false},
                          {"small 1D", kSmallThreads, 2, 1, true, false}, {"diffusive", kDTile, kDTileShared, 3, false, true},
                          {"diffusive 1D", kDTile, kDTileShared, 1, false, true}};
    const int lengths[] = {1, 2, 7, 8, 13, 14, 15, 61, 62, 64, 73, 74, 75, 123, 124, 125, 148, 200, 500, 501, 502};
    const int across[][2] = {{1, 1}, {1, 9}, {3, 5}, {8, 8}, {0, 2}, {-1, 3}, {200, 1}};
    int cases = 0;
    for (const Kind& t : kinds)
        for (int axis = 0; axis < 2; axis++)
            for (int nA : lengths)
                for (const auto& c : across) {
                    int R = 0, W = 0, ntA = 0;
                    if (t.diff)
                        dtile_shape(t.dim, nA, R, W, ntA);
                    else
                        mtile_shape(nA, R, W, ntA, t.small, t.dim);
                    const int nU = c[0] > 0 ? c[0] : W - c[0];  // a tile's row, and one column more
                    cases++;
                    if (check(t, axis, nA, nU, c[1])) {
                        std::printf("%s, axis %d, %d cells along, %d x %d across\n", t.name, axis, nA, nU, c[1]);
                        return 1;
                    }
                }
    std::printf("%d tilings\n", cases);
    return 0;
}
