// Every tile of an image comes once in strip order, and strip_pixels is the
// running sum of the tiles' on-screen pixels.  Prints the mismatches.
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
    }
    printf("%d mismatches\n", bad);
    return bad != 0;
}
