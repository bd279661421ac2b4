// Checks mafx::col_tile for every column length up to 5000 (the launch takes those with a schedule), both
// value types, narrow and wide meshes: the tile fits LDS, the group is whole waves of at most 512 lanes,
// and where the halves run one after the other the lanes cover every output.
#include <cstdio>

#include "mix_tiles.hpp"

int main() {
    int bad = 0, halves = 0;
    for (int M = 1; M <= 5000; ++M)
        for (size_t csz : {8, 16})
            for (int hx : {2, 7, 101, 1025, 8193})
                for (int64_t fill : {3, 768}) {
                    const mafx::ColTile t = mafx::col_tile(csz, M, hx, fill);
                    if (t.W == 0) {
                        const bool one = mafx::mix_lds_bytes(csz, M, 3) <= mafx::kLdsMax && 3 * M <= mafx::kColAcc * 512;
                        if (one) bad = std::printf("FAIL M=%d csz=%zu: a column fits, no tile\n", M, csz);
                        continue;
                    }
                    const bool shape = t.block >= 64 && t.block <= 512 && t.block % 64 == 0 &&
                                       mafx::mix_lds_bytes(csz, M, 3 * t.NH * t.W) <= mafx::kLdsMax;
                    halves += t.NH == 1;
                    const bool covers = t.NH == 2 || 3 * M * t.W <= mafx::kColAcc * t.block;
                    if (!shape || !covers)
                        bad = std::printf("FAIL M=%d csz=%zu hx=%d: W=%d NH=%d block=%d, %d outputs\n", M, csz, hx, t.W, t.NH,
                                          t.block, 3 * M * t.W);
                }
    if (halves == 0) bad = std::printf("FAIL no length takes its halves one after the other\n");
    if (!bad) std::printf("ok\n");
    return bad ? 1 : 0;
}
