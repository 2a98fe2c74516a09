// Which strip (64 rows x bn columns) of an output each block of the strip kernel takes. Host and device share
// the mapping; no runtime calls, so a CPU test can walk it.
#ifndef G4_STRIP_GRID_H
#define G4_STRIP_GRID_H

#include <cstdint>

namespace g4 {

// Blocks go to the 8 XCDs round robin. XCD x takes row group x % xm and column group x / xm of xm x (8 / xm)
// groups, so that its strips share its L2's copy of a few rows and columns. xm 0: the strips in turn.
struct StripGrid {
    int tiles_m, tiles_n, xm, group_m, blocks;
};

// The strip of a block; false for a block past its group's strips.
constexpr bool strip_tile(int block, int tiles_m, int tiles_n, int xm, int group_m, int &tm, int &tn) {
    if (xm > 0) {
        const int xcd = block & 7, idx = block >> 3;
        const int group_n = (tiles_n * xm + 7) >> 3;  // ceil(tiles_n / (8 / xm))
        tm = (xcd & (xm - 1)) * group_m + idx % group_m;
        tn = xcd / xm * group_n + idx / group_m;
    } else {
        tm = block % tiles_m;
        tn = block / tiles_m;
    }
    return tm < tiles_m && tn < tiles_n;
}

// The grouping that reads the fewest bytes per XCD (rows K bytes, columns K * bits / 8) among those whose group
// fits the `cus` / 8 CUs of an XCD once: a 33rd strip on one XCD is a second round for the whole call (f32 x,
// 281 x 1536 -> 2048 13.8 us with 33 strips on an XCD, 9.6 with 30; 513 x 256 -> 1024 10.7, 7.6). If none fits, the
// strips in turn, which fit an XCD whenever they fit the chip (1132 x 5632 -> 884 31.4 us with 36 on an XCD, 21.7
// in turn).
inline StripGrid strip_grid(int bits, int m, int n, int bn, int cus) {
    StripGrid G{(m + 63) / 64, (n + bn - 1) / bn, 0, 1, 0};
    G.blocks = G.tiles_m * G.tiles_n;
    int64_t least = INT64_MAX;
    for (int xm = 1; xm <= 8; xm *= 2) {
        const int64_t gm = (G.tiles_m + xm - 1) / xm, gn = ((int64_t)G.tiles_n * xm + 7) / 8;
        const int64_t bytes = gm * 64 * 8 + gn * bn * bits;
        if (gm * gn > cus / 8 || bytes >= least) continue;
        least = bytes;
        G.xm = xm, G.group_m = (int)gm, G.blocks = (int)(8 * gm * gn);
    }
    return G;
}

}  // namespace g4

#endif  // G4_STRIP_GRID_H
