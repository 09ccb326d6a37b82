// Every tile of an image comes once in strip order and in the denoisers', and
// strip_pixels is the running sum of the tiles' on-screen pixels.  Prints the mismatches.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "vpt_tiles.h"

int main(int argc, char** argv)
{
    int bad = 0;
    for (int a = 1; a + 1 < argc; a += 2) {
        const int W = atoi(argv[a]), H = atoi(argv[a + 1]);
        const uint32_t tx = (uint32_t)(W + 15) / 16u, ty = (uint32_t)(H + 15) / 16u;
        std::vector<int> seen(tx * ty, 0);
        size_t sum = 0;
        for (uint32_t t = 0; t < tx * ty; t++) {
            bad += vpt::strip_pixels(t, W, H) != sum;
            const vpt::TileXY p = vpt::strip_tile(t, tx, ty);
            if (p.x >= tx || p.y >= ty || seen[p.y * tx + p.x]++) {
                bad++;
                continue;
            }
            const int x1 = (int)p.x * 16 + 16, y1 = (int)p.y * 16 + 16;
            sum += (size_t)((x1 < W ? x1 : W) - (int)p.x * 16) * (size_t)((y1 < H ? y1 : H) - (int)p.y * 16);
        }
        bad += vpt::strip_pixels(tx * ty, W, H) != sum || sum != (size_t)W * H;

        // the denoisers' order of their 32x8 tiles
        const uint32_t dx = (uint32_t)(W + 31) / 32u, dy = (uint32_t)(H + 7) / 8u;
        for (int narrow = 0; narrow < 2; narrow++) {
            std::vector<int> once(dx * dy, 0);
            for (uint32_t t = 0; t < dx * dy; t++) {
                const vpt::TileXY p = vpt::pass_tile_at(t, dx, dy, narrow != 0);
                bad += p.x >= dx || p.y >= dy || once[p.y * dx + p.x]++;
            }
        }
    }
    printf("%d mismatches\n", bad);
    return bad != 0;
}
