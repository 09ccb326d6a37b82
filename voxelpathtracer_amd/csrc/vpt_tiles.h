// The order in which screen passes take their tiles.
//
// Each XCD has its own CUs and L2, and takes a contiguous eighth of the tiles
// (xcd_remap), so that its L2 serves one region of the world.  The eighths
// are vertical strips, not horizontal bands: a frame's cost varies with the
// height on the screen (sky rays leave in a few steps and the denoisers pass
// sky through, rays near the horizon walk far), so a band's XCD could have
// 1.7 times the mean work and the launch waited for it, while columns differ
// by a fifth.  Each strip is taken from its bottom row up: the sky's short
// blocks then come last and level out the end of the launch.  384x128x384
// terrain at 1920x1080, bands / strips from the top / from the bottom: trace
// passes 389 / 305 / 300 us, SVGF frame 958 / 853 / 761, shadow denoise
// 317 / 264 / 229, pipeline frame 1675 / 1475 / 1326.  Strips of a 24th or a
// 40th dealt in turn were no better (300, 762, 222, 1345).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "vpt/vpt_numerics.h"

namespace vpt {

struct TileXY {
    uint32_t x, y;
};

// Width of a strip in tiles, of an image tx tiles wide; an image narrower
// than 8 tiles has one strip per tile column.
VPT_HD uint32_t strip_width(uint32_t tx) { return tx >= 8u ? tx / 8u : 1u; }

// The t-th of tx x ty tiles in strip order: strips from left to right (the
// last one also takes the remaining columns), each row by row.
VPT_HD TileXY strip_tile(uint32_t t, uint32_t tx, uint32_t ty)
{
    const uint32_t sw = strip_width(tx), last = tx / sw - 1u;
    const uint32_t k = t / (sw * ty), s = k < last ? k : last;
    const uint32_t r = t - s * sw * ty, width = s == last ? tx - s * sw : sw;
    return TileXY{s * sw + r % width, r / width};
}

// The denoisers' order.  Bands, row by row from the bottom, where every tile has
// a CU to itself (256 of them): no XCD's load is left to level there.  SVGF
// frame of 200 x 91 (84 tiles of 32 x 8) in strips / bands 113 / 103 us, 482
// x 110 (224) 121 / 96, 640 x 91 (240) 99 / 102; above, 900 x 91 (348) 104 /
// 112, 482 x 180 (368) 109 / 114, 482 x 360 124 / 138.
// A last column a few pixels wide (`narrow`) is not part of the strips; its
// tiles come one after each row's worth of the others.  As a strip of its own
// its blocks lay on one XCD, took their branches alike and waited for the same
// instructions (pre-spatial pass of 482 x 91: 13.2 us, 6.8 where they were
// spread): SVGF frame of 260 x 241 136 -> 112 us, 1924 x 1080 752 -> 732.
constexpr uint32_t kBandTiles = 256u;

VPT_HD TileXY pass_tile_at(uint32_t t, uint32_t tx, uint32_t ty, bool narrow)
{
    if (tx * ty <= kBandTiles) return TileXY{t % tx, t / tx};
    if (narrow && tx > 1u) {
        const uint32_t row = t / tx;
        if (t % tx == tx - 1u) return TileXY{tx - 1u, row};
        return strip_tile(t - row, tx - 1u, ty);
    }
    return strip_tile(t, tx, ty);
}

// Pixels of the first t 16x16 tiles of a W x H image in strip order.
inline size_t strip_pixels(uint32_t t, int W, int H)
{
    const uint32_t tx = (uint32_t)(W + 15) / 16u, ty = (uint32_t)(H + 15) / 16u;
    const uint32_t sw = strip_width(tx), last = tx / sw - 1u;
    const uint32_t k = t / (sw * ty), s = k < last ? k : last;
    const uint32_t r = t - s * sw * ty, width = s == last ? tx - s * sw : sw;
    // pixels of the first n tiles along an axis of `size` pixels
    auto upto = [](uint32_t n, int size) { return 16u * n < (uint32_t)size ? (size_t)16u * n : (size_t)size; };
    const size_t x0 = upto(s * sw, W), y0 = upto(r / width, H);
    return x0 * (size_t)H + (upto(s * sw + width, W) - x0) * y0 +
           (upto(s * sw + r % width, W) - x0) * (upto(r / width + 1u, H) - y0);
}

}  // namespace vpt
