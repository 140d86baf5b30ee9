// pt_model.h — model tables and per-agent device functions of the daily loop.
//
// The functions here are the per-thread bodies of the reference's device
// functions (citations relative to PandemicThrust/PandemicThrust/), written
// for gfx950.  Floating point follows the reference's single-precision
// operation order; the library is built with -ffp-contract=off and IEEE
// division so that results are bit-identical to the reference semantics.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pt {

constexpr int kTypes = 14;
constexpr int kHhRows = 9;
constexpr int kChildRows = 5;
constexpr int kAgeAdult = 5;
constexpr int kCulmination = 10;
constexpr int kFirstErrandRow = 9;
constexpr int kTypeAfterschool = 8;
constexpr int kTypePreschool = 3;
constexpr int kWdHours = 2, kWeHours = 10;
constexpr int kWdErrands = 2, kWeErrands = 3;
constexpr int kContactsWd = 8, kContactsWe = 5;
enum ContactType : int { CT_NONE = 0, CT_WORKPLACE, CT_SCHOOL, CT_ERRAND, CT_AFTERSCHOOL, CT_HOME };
constexpr uint8_t kRecovered = 0, kSusceptible = 1, kInfected = 2;
constexpr uint8_t kDayNone = 255, kGenNone = 255;

// Model tables of one simulation (also stored in checkpoints: the layout is
// part of their format).
struct ModelData {
    float hh_cdf[kHhRows];
    int32_t hh_adults[kHhRows];
    int32_t hh_children[kHhRows];
    float child_cdf[kChildRows];
    float wp_pdf[kTypes];
    int32_t wp_count[kTypes];
    int32_t wp_offset[kTypes];
    int32_t wp_max[kTypes];
    float wd_pdf[kTypes];
    float we_pdf[kTypes];
    int32_t wd_assign[4][2];
    int32_t we_assign[6][2];
    float shed[6][10];
    float factor[2];
    float pct;
    int32_t pad0;
    uint64_t key0, key1;  // Threefry2x64 key {SEED[0], SEED[1]}
    int32_t N, H, W;
    // Dense errand-table layout: every errand destination lies in
    // [base, W), so bucket (hour, loc) maps to hour * E + (loc - base).
    // Weekday hour 1 keeps only [wd_base1, W) (weekday_keys).
    int32_t wd_base, wd_E;
    int32_t we_base, we_E;
    int32_t wd_base1, wd_E1, wd_K;
    int32_t pad1;
    // Interventions (none in the reference; the neutral values reproduce it
    // exactly): per strain, infectious while lat <= day - infection day <
    // lat + dur (reference: 0, 10); weekday school closure [school_start,
    // school_start + school_days); shares of workplace / errand contacts
    // dropped; share of agents immune to each strain from setup.  Drop and
    // vaccination draws come from their own Threefry stream (key ikey0,
    // ikey1), so no draw of the model's stream is consumed or moved.
    int32_t lat[2], dur[2];
    int32_t school_start, school_days;
    float wp_red, er_red, vacc[2];
    int32_t drops;  // any contact can be dropped (school closure or a reduction > 0)
    int32_t pad2;
    uint64_t ikey0, ikey1;
};

// An errand walk (walk_errand_rows) prepared for evaluation without division
// or loop: the rows kFirstErrandRow..kTypes-1 with a non-zero pdf, the pdfs
// scaled by 2^32 so that the walk starts from (float)u itself.
constexpr int kWalkRows = 4;
struct ErrandWalk {
    float pdf[kWalkRows];    // row pdf * 2^32
    float rcp[kWalkRows];    // 1 / pdf, rounded to nearest
    float count[kWalkRows];  // locations of the row
    int32_t offset[kWalkRows];
};

// The same as a table of the rows, for kernels that keep it in LDS
// (LdsWalk): row i ends at threshold[i]; hi + lo = the pdfs before it.
struct WalkRow {
    float hi, lo, rcp, pdf;
    float count;
    uint32_t last;  // bits of the largest float below count
    int32_t offset, pad;
};
struct WalkTable {
    WalkRow row[kWalkRows];
    float threshold[kWalkRows];
};

// The model with its prepared walks: resident in device memory, one copy per
// simulation.
struct Model : ModelData {
    ErrandWalk wd_walk, we_walk;
    WalkTable wd_table, we_table;
};

// ---------------- Threefry (Salmon et al., SC'11) ----------------
__host__ __device__ __forceinline__ uint64_t rotl64(uint64_t x, unsigned n) {
    return (x << n) | (x >> (64 - n));
}
__host__ __device__ __forceinline__ uint32_t rotl32(uint32_t x, unsigned n) {
    return (x << n) | (x >> (32 - n));
}

// Threefry2x64, 20 rounds, counter {c, c}: the reference always passes the
// same 64-bit offset in both counter words (e.g. PandemicSim.cu:2340).
struct U4 { uint32_t w[4]; };

// Word i (0..3) of a draw, selected without dynamic indexing (an indexed
// read of a register array is placed in scratch memory).
__host__ __device__ __forceinline__ uint32_t word(const U4& u, int i) {
    return i == 0 ? u.w[0] : (i == 1 ? u.w[1] : (i == 2 ? u.w[2] : u.w[3]));
}
// 64-bit rotate left by a constant 0 < n < 64 as two 32-bit funnel shifts
// (v_alignbit_b32): hi' = (hi:lo) >> (32 - n), lo' = (lo:hi) >> (32 - n)
// for n < 32; halves swapped first for n >= 32.
template <unsigned n>
__device__ __forceinline__ uint64_t rotl64c(uint64_t x) {
    const uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
    if (n == 32) return ((uint64_t)lo << 32) | hi;
    const uint32_t a = n < 32 ? hi : lo, b = n < 32 ? lo : hi;
    constexpr unsigned s = 32u - (n & 31u);
    return ((uint64_t)__builtin_amdgcn_alignbit(a, b, s) << 32) | __builtin_amdgcn_alignbit(b, a, s);
}

// 64-bit add as a 32-bit add with carry out and one with carry in: the
// v_lshl_add_u64 the compiler picks takes longer than the two (50M draws:
// 243 us with it, 198 us with these).
__device__ __forceinline__ uint64_t add64(uint64_t a, uint64_t b) {
    uint32_t lo, hi;
    asm("v_add_co_u32 %0, vcc, %2, %4\n\tv_addc_co_u32 %1, vcc, %3, %5, vcc"
        : "=&v"(lo), "=v"(hi)
        : "v"((uint32_t)a), "v"((uint32_t)(a >> 32)), "v"((uint32_t)b), "v"((uint32_t)(b >> 32))
        : "vcc");
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ U4 draw4(uint64_t c, uint64_t k0, uint64_t k1) {
    const uint64_t k2 = 0x1BD11BDAA9FC1A22ull ^ k0 ^ k1;
    uint64_t x0 = c + k0, x1 = c + k1;
#define PT_R(n) x0 = add64(x0, x1); x1 = rotl64c<n>(x1); x1 ^= x0;
#define PT_INJ(a, b, s) x0 = add64(x0, a); x1 = add64(x1, b + (uint64_t)(s));
    PT_R(16) PT_R(42) PT_R(12) PT_R(31) PT_INJ(k1, k2, 1)
    PT_R(16) PT_R(32) PT_R(24) PT_R(21) PT_INJ(k2, k0, 2)
    PT_R(16) PT_R(42) PT_R(12) PT_R(31) PT_INJ(k0, k1, 3)
    PT_R(16) PT_R(32) PT_R(24) PT_R(21) PT_INJ(k1, k2, 4)
    PT_R(16) PT_R(42) PT_R(12) PT_R(31) PT_INJ(k2, k0, 5)
#undef PT_R
#undef PT_INJ
    U4 r;
    // Union layout of the reference (u32 word 2i = low half of output i).
    r.w[0] = (uint32_t)x0;
    r.w[1] = (uint32_t)(x0 >> 32);
    r.w[2] = (uint32_t)x1;
    r.w[3] = (uint32_t)(x1 >> 32);
    return r;
}

// Threefry2x32, 20 rounds (the weekend errand-contact draw,
// PandemicSim.cu:1895-1901).
__device__ __forceinline__ void draw2x32(uint32_t c, uint32_t k0, uint32_t k1, uint32_t out[2]) {
    const uint32_t k2 = 0x1BD11BDAu ^ k0 ^ k1;
    uint32_t x0 = c + k0, x1 = c + k1;
#define PT_R(n) x0 += x1; x1 = rotl32(x1, n); x1 ^= x0;
#define PT_INJ(a, b, s) x0 += a; x1 += b + (uint32_t)(s);
    PT_R(13) PT_R(15) PT_R(26) PT_R(6) PT_INJ(k1, k2, 1)
    PT_R(17) PT_R(29) PT_R(16) PT_R(24) PT_INJ(k2, k0, 2)
    PT_R(13) PT_R(15) PT_R(26) PT_R(6) PT_INJ(k0, k1, 3)
    PT_R(17) PT_R(29) PT_R(16) PT_R(24) PT_INJ(k1, k2, 4)
    PT_R(13) PT_R(15) PT_R(26) PT_R(6) PT_INJ(k2, k0, 5)
#undef PT_R
#undef PT_INJ
    out[0] = x0;
    out[1] = x1;
}

// (float)u / UNSIGNED_MAX: the divisor converts to 2^32 in float, so this
// is an exact scaling of the round-to-nearest conversion.
__host__ __device__ __forceinline__ float unit_float(uint32_t u) { return (float)u / 4294967296.0f; }

// ---------------- setup draws ----------------
// device_setup_fishHouseholdType (PandemicSim.cu:2360-2371)
__device__ __forceinline__ int fish_household(const Model& M, uint32_t r) {
    const float y = unit_float(r);
    int row = 0;
    while (y > M.hh_cdf[row] && row < kHhRows - 1) row++;
    return row;
}

// device_setup_fishWorkplace (PandemicSim.cu:2374-2399)
// row: the type of the workplace.  The reference's loop, while (pdf[row] < y)
// y -= pdf[row++], over every row with selects: the rows are read as scalars.
__host__ __device__ __forceinline__ int32_t fish_workplace(const ModelData& M, uint32_t r, int& row) {
    float y = unit_float(r);
    row = 0;
    bool go = true;
#pragma unroll
    for (int t = 0; t < kTypes - 1; ++t) {
        go = go & (M.wp_pdf[t] < y);
        const float rest = y - M.wp_pdf[t];
        y = go ? rest : y;
        row = go ? t + 1 : row;
    }
    const float frac = y / M.wp_pdf[row];
    const int type_count = M.wp_count[row];
    int bn = (int)(frac * (float)type_count);
    if (bn >= type_count) bn = type_count - 1;
    return bn + M.wp_offset[row];
}

// device_setup_fishSchoolAndAge (PandemicSim.cu:2402-2442)
__host__ __device__ __forceinline__ int32_t fish_school_and_age(const ModelData& M, uint32_t r, uint8_t& age, int& type) {
    const float y = unit_float(r);
    int row = 0;
#pragma unroll
    for (int t = 0; t < kChildRows - 1; ++t) row += y > M.child_cdf[t];  // (the cdf ascends)
    type = row + kTypePreschool;
    float frac;
    if (row == 0) {
        frac = y / M.child_cdf[0];
    } else {
        const float pdf_here = M.child_cdf[row] - M.child_cdf[row - 1];
        const float y_here = y - M.child_cdf[row - 1];
        frac = y_here / pdf_here;
    }
    const int type_count = M.wp_count[type];
    int bn = (int)(frac * (float)type_count);
    if (bn >= type_count) bn = type_count - 1;
    age = (uint8_t)row;
    return bn + M.wp_offset[type];
}

// device_setup_assignWorkplaceOrSchool (PandemicSim.cu:2445-2457): the
// workplace or school, its contacts per day (workplace_max_contacts, from the
// type at hand instead of a search), and the age.
__host__ __device__ __forceinline__ int32_t assign_workplace(const ModelData& M, uint32_t r, bool adult, uint8_t& age,
                                                             int& contacts) {
    int type;
    int32_t wp;
    if (adult) {
        wp = fish_workplace(M, r, type);
        age = kAgeAdult;
    } else {
        wp = fish_school_and_age(M, r, age, type);
    }
    // A walk that ends on a type without workplaces gives the one before its
    // offset, the last of the type before.
    contacts = M.wp_max[M.wp_count[type] > 0 ? type : type - 1];
    return wp;
}

// ---------------- errand draws ----------------
// The reference's errand walks go through the type rows from kFirstErrandRow,
//     while (frac > pdf[row] && row < kTypes - 1) { frac -= pdf[row]; row++; }
//     bn = (int)(frac / pdf[row] * count[row])   (at most count[row] - 1)
// from frac = (float)u / 2^32.  Here the same floats are reached with 30
// instructions instead of 41 (VALU bound: 50M agents' weekday keys 236 ->
// 184 us, weekend keys 623 -> 511 us, with the adds of draw4):
// - Everything is scaled by 2^32, a power of two, so no rounding changes.
// - A row with pdf 0 is never where the walk stops (frac > 0 behind it), so
//   it is left out; the 4 remaining rows are three compares and selects.  A
//   remainder exceeds its row's pdf only if the rows before were passed, so
//   the compares need no chaining.
// - frac / pdf: with rcp = RN(1 / pdf), q0 = RN(frac rcp) is within one ulp of
//   the quotient, its remainder is exact in one fma and q = RN(q0 + rem rcp)
//   is the correctly rounded quotient (Markstein, 1990); no step over- or
//   underflows here (2^0 <= frac <= 2^32, or frac = 0).
// - The result is clamped below count as a float (counts here are below
//   2^24, so exact): the largest float below count truncates to count - 1.
static_assert(kTypes - kFirstErrandRow == 5, "errand rows");

// The walk's constants in vector registers: the selects below cannot read
// them from scalar ones (their condition already takes the one scalar operand
// an instruction may have), and left to itself the compiler branches around
// the loads.  Take it outside the loop over agents.
__device__ __forceinline__ ErrandWalk pinned(const ErrandWalk& m) {
    ErrandWalk k = m;
#pragma unroll
    for (int r = 0; r < kWalkRows; ++r)
        asm volatile("" : "+v"(k.pdf[r]), "+v"(k.rcp[r]), "+v"(k.count[r]), "+v"(k.offset[r]));
    return k;
}

struct RowPick {
    float frac, pdf, rcp, count;
    int32_t offset;
};

__device__ __forceinline__ RowPick walk_errand_rows(const ErrandWalk& k, uint32_t u) {
    const float y = (float)u;
    const float r1 = y - k.pdf[0], r2 = r1 - k.pdf[1], r3 = r2 - k.pdf[2];
    const bool c1 = y > k.pdf[0], c2 = r1 > k.pdf[1], c3 = r2 > k.pdf[2];
    auto sel = [&](auto a, auto b, auto c, auto d) {
        a = c1 ? b : a;
        a = c2 ? c : a;
        return c3 ? d : a;
    };
    return RowPick{sel(y, r1, r2, r3), sel(k.pdf[0], k.pdf[1], k.pdf[2], k.pdf[3]),
                   sel(k.rcp[0], k.rcp[1], k.rcp[2], k.rcp[3]), sel(k.count[0], k.count[1], k.count[2], k.count[3]),
                   sel(k.offset[0], k.offset[1], k.offset[2], k.offset[3])};
}

// (int)(q * count), at most count - 1.
__device__ __forceinline__ int32_t location_in_row(float q, float count) {
    // (min of the bits: both are >= 0, and fminf would first quiet NaNs)
    return (int32_t)(uint32_t)__uint_as_float(min(__float_as_uint(q * count), __float_as_uint(count) - 1u));
}

__device__ __forceinline__ int32_t walk_location(const RowPick& p) {
    const float q0 = p.frac * p.rcp;
    const float q = __builtin_fmaf(__builtin_fmaf(-q0, p.pdf, p.frac), p.rcp, q0);
    return location_in_row(q, p.count) + p.offset;
}

// The walk with its row constants read from LDS by row number instead of
// selected: 15 selects and 3 subtractions less per errand, two LDS reads more
// (weekday keys of 50M agents 176 -> 148 us, weekend keys 501 -> 457 us).
// Thresholds: remainder > pdf exactly when y > the sum of the pdfs so far
// (the remainders are exact), i.e. when y exceeds that sum rounded down.  The
// remainder is y minus that sum as two exact subtractions: hi is the sum
// rounded to a multiple of 256, which y is a multiple of behind the first row
// (y > 2^31 there), so y - hi is exact, and the rest is the exact remainder.
struct LdsWalk {
    const WalkRow* row;
    float t0, t1, t2;
};
// s_row: kWalkRows rows of LDS, filled by the block (barrier after it).
__device__ __forceinline__ LdsWalk load_walk(const WalkTable& t, WalkRow* s_row) {
    constexpr int kWords = sizeof(t.row) / 4;
    if (threadIdx.x < kWords)
        reinterpret_cast<uint32_t*>(s_row)[threadIdx.x] = reinterpret_cast<const uint32_t*>(t.row)[threadIdx.x];
    return LdsWalk{s_row, t.threshold[0], t.threshold[1], t.threshold[2]};
}
__device__ __forceinline__ int32_t fish_errand_dest(const LdsWalk& k, uint32_t r) {
    const float y = (float)r;
    int i = y > k.t0 ? 1 : 0;
    i = y > k.t1 ? 2 : i;
    i = y > k.t2 ? 3 : i;
    const WalkRow w = k.row[i];
    const float frac = (y - w.hi) - w.lo;
    const float q0 = frac * w.rcp;
    const float q = __builtin_fmaf(__builtin_fmaf(-q0, w.pdf, frac), w.rcp, q0);
    return (int32_t)(uint32_t)__uint_as_float(min(__float_as_uint(q * w.count), w.last)) + w.offset;
}

// An adult's weekday errand (device_fishAfterschoolOrErrandDestination_weekday,
// PandemicSim.cu:2909-2947) or a weekend errand
// (device_fishWeekendErrandDestination, :1017-1044); a child's weekday
// destination is its after-school site.
__device__ __forceinline__ int32_t fish_errand_dest(const ErrandWalk& k, uint32_t r) {
    return walk_location(walk_errand_rows(k, r));
}
__device__ __forceinline__ int32_t fish_afterschool(const Model& M, uint32_t r) {
    return location_in_row(unit_float(r), (float)M.wp_count[kTypeAfterschool]) + M.wp_offset[kTypeAfterschool];
}

// Weekday errand destinations of one person from its two draws
// (device_assignAfterschoolOrErrandDests_weekday, PandemicSim.cu:2950-2969),
// returned as locations (hour 1's W offset is not added).
template <class Walk>
__device__ __forceinline__ void weekday_dests(const Model& M, const Walk& k, uint32_t r1, uint32_t r2,
                                              bool adult, int32_t& d1, int32_t& d2) {
    // A wave holds adults and children alike, so every lane does both and
    // selects.
    const int32_t e1 = fish_errand_dest(k, r1), e2 = fish_errand_dest(k, r2), a = fish_afterschool(M, r1);
    d1 = adult ? e1 : a;
    d2 = adult ? e2 : a;
}

// ---------------- interventions ----------------

// Sixteen-bit uniform of contact slot c (0..7) from one draw of the
// intervention stream.
__host__ __device__ __forceinline__ float drop_uniform(const U4& x, int c) {
    return (float)((x.w[c >> 1] >> (16 * (c & 1))) & 0xFFFFu) * (1.0f / 65536.0f);
}

// Contact interventions for one infector, applied after its contacts are
// chosen: on a weekday inside the closure window school and after-school
// contacts are dropped; a workplace (errand) contact is dropped when its
// slot's uniform is below the workplace (errand) reduction.  A dropped slot
// becomes (victim -1, CT_NONE); the infector's normalising contact count is
// left as it was, so closing a place removes its transmission rather than
// moving it to the remaining contacts.  Mc is the infector's contact counter.
__device__ __forceinline__ void apply_drops(const Model& M, int day, bool weekend, uint64_t Mc, int C,
                                            int32_t (&vic)[8], int (&typ)[8]) {
    if (!M.drops) return;
    const U4 x = draw4(Mc, M.ikey0, M.ikey1);
    const bool closed = !weekend && day >= M.school_start && day < M.school_start + M.school_days;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        if (c >= C) break;
        const int t = typ[c];
        bool drop = false;
        if (t == CT_SCHOOL || t == CT_AFTERSCHOOL)
            drop = closed;
        else if (t == CT_WORKPLACE)
            drop = drop_uniform(x, c) < M.wp_red;
        else if (t == CT_ERRAND)
            drop = drop_uniform(x, c) < M.er_red;
        if (drop) {
            vic[c] = -1;
            typ[c] = CT_NONE;
        }
    }
}

// Counter of agent i's vaccination draw in the intervention stream (kept
// apart from the contact counters by the top bit).
__host__ __device__ __forceinline__ uint64_t vaccination_counter(int64_t i) { return (1ull << 63) | (uint64_t)i; }

// Weekday errand-table keys of one person.  Hour 0 spans every destination
// in [wd_base, W): key d1 - wd_base.  In hour 1 a child stays at its
// after-school site and makes no contacts there (contact profile 3 has none
// in hour 1, PandemicSim.cu:454-455), and adults only reach [wd_base1, W)
// (wd_base1 = the lowest destination fish_weekday_dest can give an adult), so
// no infector ever draws from an hour-1 bucket below wd_base1.  Hour 1 keeps
// [wd_base1, W) at keys wd_E + (d2 - wd_base1); every hour-1 entry below it
// goes to the last bucket wd_K - 1, which nobody queries.  Returns false for
// a destination outside [wd_base, W) (the keys are then clamped in range).
// (Bitwise & and selects, not && and ?: over loads: the compiler would
// otherwise branch around the model reads.)
__device__ __forceinline__ bool weekday_keys(const Model& M, int32_t d1, int32_t d2, uint32_t& k0, uint32_t& k1) {
    const int32_t E = M.wd_E, E1 = M.wd_E1, K = M.wd_K, base = M.wd_base, base1 = M.wd_base1, W = M.W;
    const int32_t l1 = d1 - base, l2 = d2 - base1;
    const bool ok = ((uint32_t)l1 < (uint32_t)E) & (d2 >= base) & (d2 < W);
    k0 = (uint32_t)min(max(l1, 0), E - 1);
    const uint32_t hour1 = (uint32_t)(E + min(l2, E1 - 1));
    k1 = l2 >= 0 ? hour1 : (uint32_t)(K - 1);
    return ok;
}

// u % kWeHours without the quarter-rate 32-bit multiplies: 65536 = 6 (mod
// 10), so u = 6 hi + lo (mod 10) < 458,746, whose quotient by 10 is exact in
// single precision (t / 10 + 0.05 is at least 0.05 from a whole number, the
// rounding errors are below 0.01).
__device__ __forceinline__ int mod_hours(uint32_t u) {
    static_assert(kWeHours == 10, "65536 = 6 (mod 10)");
    const uint32_t hi = u >> 16, t = (hi << 2) + ((hi << 1) + (u & 0xFFFFu));
    const uint32_t q = (uint32_t)__builtin_fmaf((float)t, 0.1f, 0.05f);
    return (int)(t - ((q << 3) + (q << 1)));
}
__device__ __forceinline__ int next_hour(int h) { return h == kWeHours - 1 ? 0 : h + 1; }

// device_generateWeekendErrands (PandemicSim.cu:980-1014): three distinct
// hours and their destinations.
template <class Walk>
__device__ __forceinline__ void weekend_errands(const Model& M, const Walk& k, uint64_t off, int32_t hour[3],
                                                int32_t loc[3]) {
    const U4 a = draw4(off, M.key0, M.key1);
    const U4 b = draw4(off + 1, M.key0, M.key1);
    const int h1 = mod_hours(a.w[0]);
    int h2 = mod_hours(a.w[1]);
    h2 = h2 == h1 ? next_hour(h2) : h2;
    int h3 = mod_hours(a.w[2]);
    // while (h3 == h1 || h3 == h2) h3 = (h3 + 1) % kWeHours, unrolled: two
    // forbidden hours end it within two steps.
    h3 = ((h3 == h1) | (h3 == h2)) ? next_hour(h3) : h3;
    h3 = ((h3 == h1) | (h3 == h2)) ? next_hour(h3) : h3;
    hour[0] = h1;
    hour[1] = h2;
    hour[2] = h3;
    loc[0] = fish_errand_dest(k, a.w[3]);
    loc[1] = fish_errand_dest(k, b.w[0]);
    loc[2] = fish_errand_dest(k, b.w[1]);
}

// device_getWorkplaceMaxContacts (PandemicSim.cu:3492-3511)
__host__ __device__ __forceinline__ int workplace_max_contacts(const ModelData& M, int32_t loc) {
    const int id = loc % M.W;
    int t = 0, off, cnt, mx;
    do {
        off = M.wp_offset[t];
        cnt = M.wp_count[t];
        mx = M.wp_max[t];
        t++;
    } while (id >= off + cnt && t < kTypes);
    return mx;
}

// device_calculateInfectionProbability (PandemicSim.cu:2307-2326)
__device__ __forceinline__ float infection_probability(const Model& M, int profile, int dd, int strain, int kval_sum) {
    if (kval_sum == 0) kval_sum = 1;
    const float alpha = M.shed[profile][dd];
    const float avg = alpha * M.factor[strain];
    return avg / (float)kval_sum;
}

// device_getInfectionProfile (PandemicSim.cu:3974-3988)
__device__ __forceinline__ uint32_t infection_profile(const Model& M, uint32_t r) {
    uint32_t prof = r % 3u + kInfected;
    if (unit_float(r) > M.pct) prof += 3;
    return prof;
}

}  // namespace pt
