// Counting keys of agent pairs (csrc/pt_count.h), on the host: destinations
// around the edges of each hour, where a key below the bucket count may be
// another hour's bucket.
#include <cstdio>

#include "pt_count.h"

using namespace pt;

int main() {
    int cases = 0, bad = 0;
    const WeekdayHours H{40, 75, 60, 25};  // hour 0: [40, 100), hour 1: [75, 100)
    const int32_t at[] = {-1, 0, 39, 40, 41, 74, 75, 76, 99, 100, 101, 124, 125, 2147483647};
    for (int32_t a0 : at)
        for (int32_t b0 : at)
            for (int32_t a1 : at)
                for (int32_t b1 : at)
                    for (int m = 0; m < 8; ++m) {
                        const bool two = m & 1;
                        const bool adult[2] = {(m & 2) != 0, two && (m & 4)};
                        const int32_t d1[2] = {a0, b0}, d2[2] = {a1, b1};
                        bool want = true;
                        for (int i = 0; i < 1 + two; ++i) {
                            want = want && d1[i] >= 40 && d1[i] < 100;
                            if (adult[i]) want = want && d2[i] >= 75 && d2[i] < 100;
                        }
                        uint32_t k0[2], k1[2];
                        const bool ok = weekday_pair_keys(H, d1, d2, adult, two, k0, k1);
                        bool good = ok == want;
                        for (int i = 0; i < 2 && ok; ++i) {
                            good = good && k0[i] == (i == 0 || two ? (uint32_t)(d1[i] - 40) : kNoKey);
                            good = good && k1[i] == (adult[i] ? 60u + (uint32_t)(d2[i] - 75) : kNoKey);
                        }
                        ++cases;
                        bad += !good;
                    }
    // Weekends: [30, 80) in each of ten hours.
    const int32_t wat[] = {-5, 29, 30, 31, 79, 80, 130, 2147483647};
    for (int32_t a : wat)
        for (int32_t b : wat)
            for (int e = 0; e < 3; ++e)
                for (int h = 0; h < 10; ++h)
                    for (int two = 0; two < 2; ++two) {
                        int32_t hour[2][3] = {{1, 2, 3}, {7, 8, 9}}, loc[2][3] = {{30, 45, 79}, {31, 30, 78}};
                        hour[0][e] = hour[1][e] = h;
                        loc[0][e] = a;
                        loc[1][e] = b;
                        const bool want = a >= 30 && a < 80 && (!two || (b >= 30 && b < 80));
                        uint32_t k[2][3];
                        const bool ok = weekend_pair_keys(30, 50u, hour, loc, two != 0, k);
                        bool good = ok == want;
                        for (int i = 0; i < 1 + two && ok; ++i)
                            for (int q = 0; q < 3; ++q)
                                good = good && k[i][q] == (uint32_t)(hour[i][q] * 50 + loc[i][q] - 30);
                        ++cases;
                        bad += !good;
                    }
    printf("%d cases, %d wrong\n", cases, bad);
    return bad ? 1 : 0;
}
