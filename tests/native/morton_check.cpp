// Check of morton_place and morton_ranks2 (gt_common.h) against dealing the bits of the index to the
// axes one after the other, for every grid of at most 14 bits and for long ones.
// prints: grids, indices
#include <cstdio>

#include "gt_common.h"

int main()
{
    long grids = 0, indices = 0;
    const auto check = [&](int e0, int e1, int e2, unsigned step) {
        const int e[3] = {e0, e1, e2}, n = e0 + e1 + e2;
        grids++;
        for (unsigned long long m = 0; m < (1ull << n); m += step) {
            unsigned t[3] = {0, 0, 0}, u[3] = {0, 0, 0}, rest = (unsigned)m;
            for (int bit = 0; bit < 31; bit++)
                for (int d = 0; d < 3; d++)
                    if (bit < e[d]) {
                        t[d] |= (rest & 1u) << bit;
                        rest >>= 1;
                    }
            for (int l = 0; l < n; l++) {
                const unsigned b = ((unsigned)m >> gt::morton_place(l, e)) & 1u;
                if (l < e0)
                    u[0] |= b << l;
                else if (l < e0 + e1)
                    u[1] |= b << (l - e0);
                else
                    u[2] |= b << (l - e0 - e1);
            }
            if (t[0] != u[0] || t[1] != u[1] || t[2] != u[2]) return false;
            if (e2 == 0) {
                int v[2];
                gt::morton_ranks2((unsigned)m, e0, e1, v);
                if ((unsigned)v[0] != t[0] || (unsigned)v[1] != t[1]) return false;
            }
            indices++;
        }
        return true;
    };
    for (int a = 0; a <= 14; a++)
        for (int b = 0; a + b <= 14; b++)
            for (int c = 0; a + b + c <= 14; c++)
                if (!check(a, b, c, 1)) return 1;
    const int more[][3] = {{31, 0, 0}, {0, 31, 0}, {0, 0, 31}, {10, 10, 10}, {11, 10, 10}, {3, 25, 2}, {1, 15, 15}, {20, 0, 11}};
    for (const auto &e : more)
        if (!check(e[0], e[1], e[2], 1048573u)) return 2;
    std::printf("%ld %ld\n", grids, indices);
    return 0;
}
