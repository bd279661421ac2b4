// Sizes of the two-buffer LDS tiles of fft_mixed.hip: bytes, lanes, and the tile of the single-layer y
// column.  Plain C++ with no HIP dependency, so host tests use the same code.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace mafx {

constexpr size_t kLdsMax = 160 * 1024;

// LDS elements to allocate for n logical elements (one spare after every 32)
constexpr int lds_padded(int n) { return n + (n >> 5) + 1; }

// LDS of a tile of `lines` lines of L elements of csz bytes: two buffers, the stage twiddles w_L^t and,
// unless the kernel has no second table, the packing or split twiddles w_2L^t, t <= L
inline size_t mix_lds_bytes(size_t csz, int L, int lines, bool second = true) {
    return (2 * static_cast<size_t>(lds_padded(L * lines)) + L + (second ? L + 1 : 0)) * csz;
}

// Lanes for a tile of n elements: one per eight, in whole waves, at most 512
inline int mix_block(int64_t n) { return static_cast<int>(std::min<int64_t>(512, std::max<int64_t>(64, (n / 8 + 63) / 64 * 64))); }

// Tile of k_col for columns of M rows: W columns per group, the even and odd ky together (NH = 2) or one
// after the other (NH = 1).  Both at once while two groups fit a CU.  With NH = 1 a lane keeps up to
// kColAcc of the 3 M W outputs of the first half, so the lanes cover them rounded up: 343 rows, 1029
// outputs, take 192 lanes, since 128 hold 1024.  W == 0: no tile fits.
constexpr int kColAcc = 8;
struct ColTile {
    int W, NH, block;
};
inline ColTile col_tile(size_t csz, int M, int hx, int64_t fill) {
    for (int nh : {2, 1})
        for (int w : {4, 2, 1}) {
            const int lines = 3 * nh * w, outputs = 3 * M * w;
            const bool fits = mix_lds_bytes(csz, M, lines) <= (nh == 1 && w == 1 ? kLdsMax : size_t{56} * 1024) &&
                              (nh == 2 || outputs <= kColAcc * 512);
            if (!fits || (w > 1 && (hx + w - 1) / w < fill)) continue;
            const int cover = (outputs + 64 * kColAcc - 1) / (64 * kColAcc) * 64;
            return {w, nh, nh == 2 ? mix_block(static_cast<int64_t>(M) * lines) : cover};
        }
    return {0, 0, 0};
}

} // namespace mafx
