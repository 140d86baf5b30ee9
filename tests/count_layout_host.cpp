// Column groups of split counted layouts (csrc/pt_count.h), on the host: the
// groups of an hour cover its buckets once, and the mark words that hold a
// group's or an hour's buckets are words of the chunk's own.
#include <cstdio>

#include "pt_count.h"

using namespace pt;

static int check(int64_t N, int kpa, int32_t E, int32_t E_last, int hours) {
    CountPlan p;
    CountRep c{};
    c.K = (hours - 1) * E + E_last;
    p.reps.assign(1, c);
    p.build_split(N, kpa, E, hours, 256);
    if (!p.on) return 0;
    c = p.reps[0];
    int bad = 0;
    for (int h = 0; h < hours; ++h) {
        const GroupColumns all = hour_columns(c, h);
        const int32_t width = h == hours - 1 ? E_last : E;
        int next = all.bucket;
        for (int g = h * c.ranges; g < (h + 1) * c.ranges; ++g) {
            const GroupColumns q = group_columns(c, g);
            bad += q.hour != h || q.n > c.W || (q.n > 0 && (q.bucket != next || q.lo != next - all.bucket));
            bad += q.n > 0 && (first_mark_word(q) < 0 || end_mark_word(q) > c.qw);
            bad += q.n == 0 && first_mark_word(q) != end_mark_word(q);
            next += q.n;
        }
        bad += all.n != width || next != all.bucket + width || end_mark_word(all) > c.qw;
        if (bad) {
            printf("N %lld, hour %d of %d: E %d, last %d, %d ranges of %d: width %d, groups end at %d\n", (long long)N,
                   h, hours, E, E_last, c.ranges, c.W, all.n, next);
            return 1;
        }
    }
    return 0;
}

int main() {
    int bad = 0, plans = 0;
    // Location scales from where layouts split to where an hour needs more
    // groups than are allowed; 1,600 and 1,300 locations per scale.
    for (double s = 3.0; s < 210.0; s *= 1.013) {
        const int32_t E = (int32_t)(1600 * s), E1 = (int32_t)(1300 * s);
        for (int64_t N : {(int64_t)943, (int64_t)235417, (int64_t)50002479}) {
            bad += check(N, 2, E, E1 + 1, 2);
            bad += check(N, 3, E1, E1, 10);
            plans += 2;
        }
    }
    printf("%d layouts, %d wrong\n", plans, bad);
    return bad ? 1 : 0;
}
