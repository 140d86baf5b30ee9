// Contacts per day from the type of the workplace walk (csrc/pt_model.h),
// against the search by location, on the host: draws around every boundary of
// the walks and across the whole range, over location scales.
#include <cmath>
#include <cstdio>

#include "pt_day.h"

using namespace pt;

// The workplace types of the reference model (the order of its counts).
static ModelData model(double scale) {
    static const float pdf[14] = {0.06586f, 0.05802f, 0.30227f, 0.0048f, 0.00997f, 0.203f, 0.09736f,
                                  0.10598f, 0.00681f, 0.02599f, 0.f,     0.08749f, 0.03181f, 0.00064f};
    static const int mx[14] = {3, 3, 3, 2, 2, 3, 3, 2, 2, 2, 0, 2, 2, 2};
    static const int base[14] = {1000, 7000, 2400, 300, 100, 200, 100, 100, 300, 500, 0, 300, 400, 100};
    static const float child[5] = {0.24f, 0.47f, 0.72f, 0.85f, 1.0f};
    ModelData m{};
    for (int t = 0; t < kTypes; ++t) {
        m.wp_pdf[t] = pdf[t];
        m.wp_max[t] = mx[t];
        m.wp_count[t] = (int)std::floor(base[t] * scale + 0.5);
        if (m.wp_count[t] == 0 && base[t]) m.wp_count[t] = 1;
        m.wp_offset[t] = t ? m.wp_offset[t - 1] + m.wp_count[t - 1] : 0;
    }
    m.W = m.wp_offset[kTypes - 1] + m.wp_count[kTypes - 1];
    for (int i = 0; i < kChildRows; ++i) m.child_cdf[i] = child[i];
    return m;
}

static int64_t cases = 0, bad = 0;

static void check(const ModelData& m, uint32_t r) {
    for (int adult = 0; adult < 2; ++adult) {
        uint8_t age = 99;
        int contacts = -1;
        const int32_t wp = assign_workplace(m, r, adult != 0, age, contacts);
        ++cases;
        if (wp < 0 || wp >= m.W || contacts != workplace_max_contacts(m, wp) || (age == kAgeAdult) != (adult != 0)) {
            if (++bad < 10) printf("W %d, draw %u, adult %d: place %d, %d contacts\n", m.W, r, adult, wp, contacts);
        }
    }
}

int main() {
    for (double scale : {0.0004, 0.0011, 0.01, 0.0425, 0.3, 1.0, 21.24, 100.0}) {
        const ModelData m = model(scale);
        double cdf = 0;
        for (int t = 0; t < kTypes; ++t) {
            cdf += m.wp_pdf[t];
            for (int d = -3000; d <= 3000; ++d) {
                check(m, (uint32_t)std::llround(std::fmin(std::fmax(cdf * 4294967296.0 + d, 0.0), 4294967295.0)));
                if (t < kChildRows)
                    check(m, (uint32_t)std::llround(
                                 std::fmin(std::fmax(m.child_cdf[t] * 4294967296.0 + d, 0.0), 4294967295.0)));
            }
        }
        for (uint32_t d = 0; d < 3000; ++d) {
            check(m, d);
            check(m, ~d);
        }
        for (uint64_t r = 0; r < (1ull << 32); r += 9973) check(m, (uint32_t)r);
    }
    printf("%lld cases, %lld wrong\n", (long long)cases, (long long)bad);
    return bad ? 1 : 0;
}
