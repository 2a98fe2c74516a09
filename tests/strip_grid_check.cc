// CPU driver for the strip kernel's grid (gemma4-webgpu-engine_amd/csrc/g4_strip_grid.h): over every grid of
// up to 256 strips, each strip is one block's, and no XCD has more strips than CUs. Built and run by
// tests/test_strip_grid.py; prints "ok" and exits 0 when it holds.
#include <cstdio>
#include <vector>

#include "g4_strip_grid.h"

int main() {
    constexpr int kCus = 256;
    for (int bits = 4; bits <= 8; bits += 4)
        for (int bn = 32; bn <= 64; bn += 16)
            for (int tm = 1; tm <= kCus; ++tm)
                for (int tn = 1; tm * tn <= kCus; ++tn) {
                    const g4::StripGrid G = g4::strip_grid(bits, 64 * tm - 5, bn * tn - 3, bn, kCus);
                    std::vector<int> taken(tm * tn, 0);
                    int per_xcd[8] = {};
                    for (int b = 0; b < G.blocks; ++b) {
                        int r = -1, c = -1;
                        if (!g4::strip_tile(b, G.tiles_m, G.tiles_n, G.xm, G.group_m, r, c)) continue;
                        ++taken[c * tm + r];
                        ++per_xcd[b % 8];
                    }
                    for (int n : taken)
                        if (n != 1) return std::printf("FAIL: %d x %d strips, one taken %d times\n", tm, tn, n), 1;
                    for (int n : per_xcd)
                        if (n > kCus / 8) return std::printf("FAIL: %d x %d strips, %d on an XCD\n", tm, tn, n), 1;
                }
    std::printf("ok\n");
    return 0;
}
