// Checks mafx::wgrad_shape over batches and image sides: a wave's FP32 sum over pixels (a chunk's tiles of
// 128 pixels, shared by at least two waves) is never longer than a sum over 64 chunks of 16 x 16 tiles, nor
// its partials more, and every tile belongs to a chunk that exists.
#include <cstdio>

#include "net_shapes.hpp"

int main() {
    int bad = 0;
    long more = 0;
    for (int l = 0; l < mafx::kNetLayers && !bad; ++l)
        for (int B = 1; B <= 520; B += B < 70 ? 1 : 45)
            for (int H = 8; H <= 264; H += 8)
                for (int W = 8; W <= 264; W += 8) {
                    const mafx::WgradShape g = mafx::wgrad_shape(l, B, H, W);
                    const int total = B * g.tiles, t16 = B * ((g.h + 15) / 16) * ((g.w + 15) / 16);
                    const int co = mafx::kNetCout[l], ci = mafx::kNetCin[l];
                    const int waves = 8 / ((co > 16 ? 2 : 1) * (ci > 16 ? 2 : 1));
                    const int chain = (total + g.nchunk - 1) / g.nchunk * 128 / waves;
                    const int c16 = t16 < 64 ? t16 : 64, chain16 = (t16 + c16 - 1) / c16 * 256;
                    if (g.nchunk < 1 || g.nchunk > total || g.nchunk > mafx::kWgradGroups || chain > chain16)
                        bad = std::printf("FAIL layer %d B=%d %dx%d: %d chunks, chain %d against %d\n", l, B, H, W, g.nchunk,
                                          chain, chain16);
                    more += g.nchunk * ((co + 31) / 32) * ((ci + 31) / 32) > mafx::kWgradGroups;
                }
    if (more == 0) bad = std::printf("FAIL no size takes the longer list of chunks\n");
    if (!bad) std::printf("ok\n");
    return bad ? 1 : 0;
}
