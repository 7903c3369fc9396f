// hm_tiles.hpp -- tiles of the fused multi-species flux and of the diffusive
// flux: their shapes, and the arithmetic that places a block's threads in them.
// Host and device code without HIP types, so that a host check can run it.
#pragma once

#include <cstdint>

#include "hm_numerics.hpp"  // HM_HD

namespace hm {

// Fused midpoint and face flux of the multi-species models (k_flux_multi): a
// 256-thread block owns a tile of R consecutive midpoint faces along the axis
// by W positions across it (R W <= 256), keeps the tile's midpoint fluxes in
// LDS and outputs the R - 2 inner faces of each of its W columns.  A column of
// n_A + 3 midpoint faces (n_A + 1 output faces) takes ntA tiles of at most
// kMTileFaces output faces each, of equal length, which share two midpoint
// faces; W is as many columns as fit.
constexpr int kMTileThreads = 256;
constexpr int kMTileFaces = 62;

// small: tiles of 64 faces (k_flux_multi_small) of at most 14 output faces, so
// that the columns of a tile are a few neighbours in memory (30 instead of 14:
// 24^3 five-equation call 27.3 us instead of 26.0); a 1D patch has one column.
constexpr int kSmallThreads = 64;
constexpr int kSmallFaces = 14;

HM_HD constexpr void mtile_shape(int nA, int& R, int& W, int& ntA, bool small = false, int dim = 3) {
    const int most = small && dim > 1 ? kSmallFaces : kMTileFaces;
    ntA = (nA + 1 + most - 1) / most;
    R = (nA + 1 + ntA - 1) / ntA + 2;
    W = (small ? kSmallThreads : kMTileThreads) / R;
}

// LDS slots of a small tile's cells, (R + 5) W, and of its cells with sensor
// values, (R + 1) W; one thread of the block takes each of either.
constexpr int kSmallCells = 144;
constexpr int kSmallSensor = 80;

// First thread of the sensor cells.
HM_HD constexpr uint32_t small_sensor_first(uint32_t ncell) { return ncell > 128u ? ncell : 128u; }

// Whether every shape of a small tile (R of 3 .. kMTileFaces + 2) fits.
constexpr bool small_tiles_fit() {
    for (int dim = 1; dim <= 3; dim++)
        for (int nA = 1; nA <= 4 * kMTileFaces; nA++) {  // (R repeats beyond one tile's faces)
            int R = 0, W = 0, ntA = 0;
            mtile_shape(nA, R, W, ntA, true, dim);
            if (R * W > kSmallThreads || (R + 5) * W > kSmallCells || (R + 1) * W > kSmallSensor) return false;
            if (small_sensor_first(uint32_t((R + 5) * W)) + uint32_t((R + 1) * W) > uint32_t(kMTileThreads)) return false;
        }
    return true;
}
static_assert(small_tiles_fit(), "a small tile's cells fit its LDS slots and its block");

// Work items of the fused axis-a segment of one patch: a block of 256 per tile.
HM_HD int64_t mtile_items(int axis, const int* n, int dim, bool small = false) {
    int64_t trans = 1;  // columns: positions across the axis
    for (int b = 0; b < dim; b++)
        if (b != axis) trans *= n[b];
    int R = 0, W = 0, ntA = 0;
    mtile_shape(n[axis], R, W, ntA, small, dim);
    return int64_t(kMTileThreads) * ntA * ((trans + W - 1) / W);
}

// Tile of the diffusive flux (k_diff_flux): a block of kDTile threads takes R
// consecutive cells along the axis by W columns (R W <= kDTile) and outputs
// R - 11 faces of each column (a face takes six nodes, a node seven cells).  A
// column of n_A + 12 cells (n_A + 1 faces) takes ntA tiles of equal length that
// share eleven cells, of at most 74 faces in 2D and 3D, so that a tile has 6
// columns or more (39 of one-cell columns), of as many as the block holds in 1D.
constexpr int kDTile = 512;
constexpr int kDTileShared = 11;

HM_HD constexpr void dtile_shape(int dim, int nA, int& R, int& W, int& ntA) {
    const int most = dim == 1 ? kDTile - kDTileShared : 74;
    ntA = (nA + 1 + most - 1) / most;
    R = (nA + 1 + ntA - 1) / ntA + kDTileShared;
    W = kDTile / R;
}

// Exact division of a thread number x by d, both up to 512, as a product: m d
// exceeds 2^20 by less than d, so x m is off by less than x d < 2^20, under one
// in the quotient's last place.
HM_HD constexpr uint32_t small_div_mul(uint32_t d) { return ((1u << 20) + d - 1u) / d; }
HM_HD constexpr uint32_t small_div(uint32_t x, uint32_t m) { return (x * m) >> 20; }

// Row r and column w of thread `lane` in a tile of R rows by W columns: threads
// run along a column on axis 0 (consecutive along x), across the columns on
// axes 1 and 2.  mul: small_div_mul of R on axis 0, of W on the others.
HM_HD constexpr void tile_place(int axis, uint32_t lane, uint32_t R, uint32_t W, uint32_t mul, uint32_t& r, uint32_t& w) {
    const uint32_t first = small_div(lane, mul);
    const uint32_t rest = lane - first * (axis == 0 ? R : W);
    r = axis == 0 ? rest : first;
    w = axis == 0 ? first : rest;
}

// Column (u, v) of a tile's position w: columns run u fastest over nU by nV
// positions, the tile's first one is t0 (block-uniform), W of them per tile.
HM_HD void tile_column(uint32_t t0, uint32_t w, uint32_t W, uint32_t nU, uint32_t& u, uint32_t& v) {
    const uint32_t v0 = t0 / nU;
    u = t0 - v0 * nU + w;
    if (nU >= W) {  // at most one row on
        const bool over = u >= nU;
        v = v0 + (over ? 1u : 0u);
        u -= over ? nU : 0u;
    } else {  // u < nU + W
        const uint32_t q = small_div(u, small_div_mul(nU));
        v = v0 + q;
        u -= q * nU;
    }
}

}  // namespace hm
