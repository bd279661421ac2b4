// Layers of the warm-start network and the split of their weight gradients.  Plain C++ with no HIP
// dependency, so host tests use the same code.
#pragma once
#include <algorithm>

namespace mafx {

// (in, out) channels of the eight 3x3 convolutions in execution order, and their level: the image is
// halved that many times
constexpr int kNetLayers = 8;
constexpr int kNetCin[kNetLayers] = {8, 32, 64, 128, 256, 128, 64, 32};
constexpr int kNetCout[kNetLayers] = {32, 64, 128, 128, 64, 32, 32, 3};
constexpr int kNetLevel[kNetLayers] = {0, 1, 2, 3, 2, 1, 0, 0};

// Level size, tiles of 128 pixels (tw wide) and chunks of a layer's weight gradient.  Work-groups are
// blocks of 32 x 32 channels times chunks, kWgradGroups at most, and each chunk writes a partial of the
// layer's gradient.  The layers of 16 blocks then have 16 chunks, which on large batches makes the FP32
// sum of a wave (one of two per chunk) longer than the sum over 64 chunks of 256-pixel tiles that the
// matrix-core form replaced: at 512 films of 64 x 64, both sums modelled with random operands, its rounding
// is 1.2 times as large.  From more than four tiles a chunk on, where a wave's sum would become the longer
// one, they take 32 chunks: 0.85 to 0.9 times as large, at the same time (8 films of 192 x 184 1614 -> 1623
// us, 512 of 64 x 64 8379 -> 8383).
constexpr int kWgradGroups = 256, kWgradLongChunks = 32;
struct WgradShape {
    int h, w, tw, tiles_x, tiles, nchunk;
};
inline WgradShape wgrad_shape(int layer, int B, int H, int W) {
    WgradShape g{};
    g.h = H >> kNetLevel[layer];
    g.w = W >> kNetLevel[layer];
    g.tw = g.w <= 8 ? 8 : 16;
    const int th = 128 / g.tw;
    g.tiles_x = (g.w + g.tw - 1) / g.tw;
    g.tiles = g.tiles_x * ((g.h + th - 1) / th);
    const int blocks = ((kNetCout[layer] + 31) / 32) * ((kNetCin[layer] + 31) / 32);
    int limit = kWgradGroups / blocks;
    if (B * g.tiles > 4 * limit) limit = std::max(limit, kWgradLongChunks);
    g.nchunk = std::max(1, std::min(B * g.tiles, limit));
    return g;
}

} // namespace mafx
