// pt_day.h — daily-loop device code shared by the single-simulation engine
// (pt_sim.hip) and the replicate-batch engine (pt_batch.hip), and the host
// helpers both use.
//
// Every function here works on one simulation in its own (local) agent,
// household, workplace and bucket numbering; the batch engine reaches a
// replicate by offsetting the array pointers and passing a bucket or id
// bias.
//
// Citations are relative to PandemicThrust/PandemicThrust/ of the reference.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/pandemic/pt_abi.h"
#include "pt_model.h"
#include "pt_sort.h"

namespace pt {

// ---------------- host helpers ----------------

// Records the error text returned by pt_last_error; returns code.
int fail(int code, const char* fmt, ...);
// PT_OK when value is in range for launch setting knob (pt_launch_knob).
int check_launch(int32_t knob, int32_t value);

// Argument checks shared by the location-table entry points (pt_table.hip).
int location_table_args(const uint32_t* keys, int64_t n, int32_t n_buckets, const int32_t* people,
                        const int32_t* offsets);

// Makes `device` current for a scope and restores the caller's device.
struct DeviceScope {
    int saved = -1;
    hipError_t err = hipSuccess;
    explicit DeviceScope(int device) {
        err = hipGetDevice(&saved);
        if (err == hipSuccess) err = hipSetDevice(device);
    }
    ~DeviceScope() {
        if (saved >= 0) (void)hipSetDevice(saved);
    }
    DeviceScope(const DeviceScope&) = delete;
    DeviceScope& operator=(const DeviceScope&) = delete;
};

#define HIP_TRY(expr)                                                                              \
    do {                                                                                           \
        hipError_t e_ = (expr);                                                                    \
        if (e_ != hipSuccess) return ::pt::fail(PT_EDEVICE, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

template <class T>
int dev_alloc(T** p, int64_t count) {
    if (count <= 0) count = 1;
    if (device_malloc((void**)p, (size_t)count * sizeof(T)) != hipSuccess) {
        *p = nullptr;
        return fail(PT_ENOMEM, "hipMalloc of %lld bytes failed", (long long)(count * (int64_t)sizeof(T)));
    }
    return 0;
}

template <class T>
void dev_free(T*& p) {
    if (p) (void)hipFree((void*)p);
    p = nullptr;
}

inline int grid_for(int64_t n, int threads, int cap) {
    return (int)std::max<int64_t>(1, std::min<int64_t>((n + threads - 1) / threads, cap));
}

// Model tables of one constants row (setup_loadParameters PandemicSim.cu:313-562,
// setup_scaleSimulation :1127-1162, setup_calculateInfectionData :2828-2840)
// and the dense errand-table layout.  Returns PT_OK or PT_EINVAL.
int build_model(const pt_params* p, const int32_t seed_key[2], Model& m);

// Validates an intervention set and writes it into the model (PT_OK or
// PT_EINVAL).
int apply_interventions(const pt_interventions* iv, Model& m);

// Pairs of the queried buckets: staged by block, then compacted (counted days
// keep their lists and picks here).  One allocation while it is small: one of
// 2 MB or more costs about 25 us to make and free again (2.35M agents, set-up
// 1.20 -> 1.15 ms), but the time of a large one grows with it (1.5 GB 270 us,
// in four 4 x 36).
struct SelectionBuffers {
    uint32_t* stage_keys = nullptr;
    int32_t* stage_ids = nullptr;
    uint32_t* sel_keys = nullptr;
    int32_t* sel_ids = nullptr;
    bool one = false;
};
inline int alloc_selection(SelectionBuffers& b, int64_t staged, int64_t selected) {
    const int64_t a = (staged + 63) / 64 * 64, c = (selected + 63) / 64 * 64;
    b.one = 2 * (a + c) * (int64_t)sizeof(uint32_t) <= ((int64_t)256 << 20);
    if (!b.one)
        return dev_alloc(&b.stage_keys, staged) || dev_alloc(&b.stage_ids, staged) ||
               dev_alloc(&b.sel_keys, selected) || dev_alloc(&b.sel_ids, selected);
    if (dev_alloc(&b.stage_keys, 2 * (a + c))) return PT_ENOMEM;
    b.stage_ids = (int32_t*)(b.stage_keys + a);
    b.sel_keys = b.stage_keys + 2 * a;
    b.sel_ids = (int32_t*)(b.sel_keys + c);
    return PT_OK;
}
inline void free_selection(SelectionBuffers& b) {
    dev_free(b.stage_keys);
    if (!b.one) {
        dev_free(b.stage_ids);
        dev_free(b.sel_keys);
        dev_free(b.sel_ids);
    }
    b = SelectionBuffers();
}

// The byte arrays of `count` agents, from 1 MB each in one allocation (seven of
// 50 MB take 210 us to make, one of 350 MB 38 us; smaller ones cost below 1 us
// each, as parts of the runtime's blocks).
template <class Owner>
int alloc_agent_bytes(Owner& o, int64_t count) {
    uint8_t** const rest[6] = {&o.st_s, &o.dy_p, &o.dy_s, &o.gn_p, &o.gn_s, &o.age};
    const int64_t stride = (count + 255) / 256 * 256;
    o.one_block = stride >= ((int64_t)1 << 20);
    if (dev_alloc(&o.st_p, o.one_block ? 7 * stride : count)) return PT_ENOMEM;
    for (int k = 0; k < 6; ++k) {
        if (o.one_block)
            *rest[k] = o.st_p + (k + 1) * stride;
        else if (dev_alloc(rest[k], count))
            return PT_ENOMEM;
    }
    return PT_OK;
}
template <class Owner>
void free_agent_bytes(Owner& o) {
    dev_free(o.st_p);
    for (uint8_t** p : {&o.st_s, &o.dy_p, &o.dy_s, &o.gn_p, &o.gn_s, &o.age}) {
        if (!o.one_block) dev_free(*p);
        *p = nullptr;
    }
}

// What a contact needs of an agent, in one 8-byte record instead of five
// gathers (age, household, its two offsets, workplace): x = first person of
// the household | its size << 28 | adult << 31; y = workplace or school | its
// contacts per day << 28.  Agents and locations number below 2^28
// (pt_sim_setup; location_scaling <= 1e4), households hold at most 5 people.
struct AgentRecord {
    uint32_t x, y;
};
__device__ __forceinline__ AgentRecord make_record(int32_t hoff, int32_t hcnt, bool adult, int32_t wp, int wpd) {
    return AgentRecord{(uint32_t)hoff | ((uint32_t)hcnt << 28) | (adult ? 0x80000000u : 0u),
                       (uint32_t)wp | ((uint32_t)wpd << 28)};
}
__device__ __forceinline__ int32_t record_household(AgentRecord a) { return (int32_t)(a.x & 0x0FFFFFFFu); }
__device__ __forceinline__ int32_t record_household_size(AgentRecord a) { return (int32_t)((a.x >> 28) & 7u); }
__device__ __forceinline__ bool record_adult(AgentRecord a) { return (a.x >> 31) != 0; }
__device__ __forceinline__ int32_t record_workplace(AgentRecord a) { return (int32_t)(a.y & 0x0FFFFFFFu); }
__device__ __forceinline__ int record_workplace_contacts(AgentRecord a) { return (int)(a.y >> 28); }

// Population arrays of one simulation (local numbering).
struct PopArrays {
    uint8_t* hh_types;   // H + 1
    int32_t* hh_off;     // H + 1
    int32_t* household;  // N
    uint8_t* age;        // N
    int32_t* wp_off;     // W + 1
    int32_t* wp_people;  // N
    AgentRecord* who;    // N
    int32_t* wp_lone;    // 1: some workplace has a single person
    uint8_t *st_p, *st_s, *dy_p, *dy_s, *gn_p, *gn_s;  // N
    uint64_t *claim_p, *claim_s;                        // N
};

// K1/K2 (PandemicSim.cu:3579-3605, :2329-2357): household types into
// hh_types and the population size added to *people (device counter).
void launch_household_types(const Model* d_model, int H, uint8_t* hh_types, unsigned long long* people,
                            hipStream_t stream);

// K3-K7 (PandemicSim.cu:2573-2613, :3812-3862, :3654-3664) for a model whose
// N is set on the device: household offsets and people, workplaces and the
// workplace table, statuses, empty claim words.  tmp holds max(N, H + 1)
// uint32; ts is sized for N pairs.  Enqueued on stream, not synchronised.
// marks, if given, are 4 events recorded before the households, after them,
// after the workplaces and after the statuses.
hipError_t build_population(const Model* d_model, int64_t N, int H, int W, const PopArrays& P, uint32_t* tmp,
                            TableScratch& ts, uint64_t workplace_off, hipStream_t stream,
                            const hipEvent_t* marks = nullptr);

// ---------------- device state ----------------

constexpr int kSweepThreads = 512;
constexpr int kSweepPer = 16;                          // agents per thread (one uint4 per array)
constexpr int kSweepTile = kSweepThreads * kSweepPer;  // 8192 agents per block
constexpr int kPlanThreads = 1024;
constexpr int kContactThreads = 256;

// The reference's host-side loop counters (PandemicSim.h:73-76,
// simRandOffsetsStruct_t) kept in device memory.
struct DayState {
    int32_t day;           // current_day
    int32_t done;          // the loop has ended
    int32_t days_run;      // rows of output_infected_stats.csv produced
    int32_t n_infected;    // infected_count of the current day
    uint64_t rand_offset;  // rand_offset
    uint64_t errand_off;   // errand_randOffset of the current day
    uint64_t contact_base; // rand_offset at the contact kernel
    uint32_t n_claimed[2]; // claim-list lengths (pandemic, seasonal)
    int32_t max_days;
    int32_t fault;         // nonzero if a kernel saw data outside the model's range
    int32_t skip_full;     // the full errand-table path is idle today
    int32_t skip_subset;   // the subset errand-table path is idle today
    uint32_t n_sel;        // pairs selected into today's subset table
    uint32_t n_marked;     // errand buckets queried today
    int32_t skip_mark;     // too many infectors today for a subset table to pay off
};

// Errand tables are built either for every bucket (full) or only for the
// buckets today's infectors draw contacts from (subset); the choice is
// made on the device from the number of queried buckets.
enum TableMode : int { TABLES_AUTO = 0, TABLES_FULL = 1, TABLES_SUBSET = 2 };
constexpr int kSelThreads = 256;
constexpr int kSelPerWd = 8;   // agents per thread, weekday selection
constexpr int kSelPerWe = 4;   // agents per thread, weekend selection
constexpr int kSelAgentsWd = kSelThreads * kSelPerWd;
constexpr int kSelAgentsWe = kSelThreads * kSelPerWe;
constexpr int kSelStageWd = kSelAgentsWd * 2;  // staged pairs per weekday selection block
constexpr int kSelStageWe = kSelAgentsWe * 3;  // staged pairs per weekend selection block

// Whether a subset table pays off: fewer than 60% of the buckets queried.
__host__ __device__ __forceinline__ bool subset_pays(int64_t marked, int64_t K, int share_pct) {
    return marked * 100 < K * share_pct;
}

// Infected count up to which a day marks its queried buckets (K * pct / 100).
__host__ __device__ __forceinline__ int64_t mark_limit(int64_t K, int pct) { return K * pct / 100; }

// ---------------- wave helpers ----------------

// Scalar loads in one batch.  Left to themselves the loads of a kernel's
// arguments, the day's state and the model come one by one as the code reaches
// them, each a miss of the scalar cache, which starts cold: some ten in a row
// before a kernel's first vector load, 1 to 3 us of launches that take 6 to 20.
// First the 64-byte lines of the arguments (all inside them) ...
template <int LINES>
__device__ __forceinline__ void load_arguments() {
    static_assert(LINES == 2 || LINES == 5 || LINES == 8, "lines");
    const auto k = (const __attribute__((address_space(4))) uint32_t*)__builtin_amdgcn_kernarg_segment_ptr();
    if constexpr (LINES == 2)
        asm volatile("" ::"s"(k[0]), "s"(k[16]));
    else if constexpr (LINES == 5)
        asm volatile("" ::"s"(k[0]), "s"(k[16]), "s"(k[32]), "s"(k[48]), "s"(k[64]));
    else
        asm volatile("" ::"s"(k[0]), "s"(k[16]), "s"(k[32]), "s"(k[48]), "s"(k[64]), "s"(k[80]), "s"(k[96]), "s"(k[112]));
}
// ... then what they point to: values, and the lines of the state and model.
template <class A, class B, class C, class D>
__device__ __forceinline__ void load_together(A a, B b, C c, D d) {
    asm volatile("" ::"s"(a), "s"(b), "s"(c), "s"(d));
}
__device__ __forceinline__ void load_state_and_model(const DayState* st, const Model* M, uint32_t more) {
    static_assert(sizeof(Model) >= 21 * 64 && sizeof(DayState) >= 68, "the lines below");
    const uint32_t* d = reinterpret_cast<const uint32_t*>(st);
    const uint32_t* m = reinterpret_cast<const uint32_t*>(M);
    asm volatile("" ::"s"(more), "s"(d[1]), "s"(d[16]), "s"(m[0]), "s"(m[16]), "s"(m[32]), "s"(m[48]), "s"(m[64]), "s"(m[80]), "s"(m[96]),
                 "s"(m[112]), "s"(m[128]), "s"(m[144]), "s"(m[160]), "s"(m[176]), "s"(m[192]), "s"(m[208]), "s"(m[224]),
                 "s"(m[240]), "s"(m[256]), "s"(m[272]), "s"(m[288]), "s"(m[304]), "s"(m[320]));
}

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v, int lane) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t t = __shfl_up(v, d, 64);
        if (lane >= d) v += t;
    }
    return v;
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

// v plus the value of the lane that the DPP control names (0 where there is
// none, or in rows that ROWS leaves out).
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ uint32_t dpp_add(uint32_t v) {
    return v + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false);
}
// Inclusive scan over the lanes of a wave that is wholly active: within rows
// of 16 lanes, then lane 15 to the next row, lane 31 to the upper half.
__device__ __forceinline__ uint32_t full_wave_scan(uint32_t v) {
    v = dpp_add<0x111>(v);  // row_shr:1
    v = dpp_add<0x112>(v);
    v = dpp_add<0x114>(v);
    v = dpp_add<0x118>(v);
    v = dpp_add<0x142, 0xA>(v);  // row_bcast:15
    return dpp_add<0x143, 0xC>(v);  // row_bcast:31
}

// Sums over the 64 lanes (all active) of eight byte counters, four to a word
// (bin b in byte b; at most 16 per lane): a scan over 8 lanes on the packed
// words (a byte reaches at most 128), the rest on 16-bit fields.  out[b] = the
// total of bin b, in lane 63.
__device__ __forceinline__ void wave_sum_bins8(uint32_t lo, uint32_t hi, uint32_t (&out)[8]) {
    lo = dpp_add<0x114>(dpp_add<0x112>(dpp_add<0x111>(lo)));
    hi = dpp_add<0x114>(dpp_add<0x112>(dpp_add<0x111>(hi)));
    uint32_t w[4] = {lo & 0x00FF00FFu, (lo >> 8) & 0x00FF00FFu, hi & 0x00FF00FFu, (hi >> 8) & 0x00FF00FFu};
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = dpp_add<0x143, 0xC>(dpp_add<0x142, 0xA>(dpp_add<0x118>(w[j])));
    // w[0]: bins 0 and 2, w[1]: 1 and 3, w[2]: 4 and 6, w[3]: 5 and 7
    out[0] = w[0] & 0xFFFFu;
    out[2] = w[0] >> 16;
    out[1] = w[1] & 0xFFFFu;
    out[3] = w[1] >> 16;
    out[4] = w[2] & 0xFFFFu;
    out[6] = w[2] >> 16;
    out[5] = w[3] & 0xFFFFu;
    out[7] = w[3] >> 16;
}

// The day's errand and contact counters (PandemicSim.cu:3030-3040,
// :1409-1415, :1278-1279, :1393-1394);
// rand_offset itself moves at the day's end.
__device__ __forceinline__ void plan_offsets(DayState* st, bool weekend, int64_t N) {
    st->errand_off = st->rand_offset;
    st->contact_base = st->rand_offset + (weekend ? (uint64_t)(2 * N) : (uint64_t)(N / 2));
}

// ---------------- D1 + D2: sweep ----------------

// Bytewise on four agents per word (bit 7 of each byte of the result): x != 0
// but for its lowest bit; x <= y.
__device__ __forceinline__ uint32_t bytes_infected(uint32_t x) {
    const uint32_t t = x & 0xFEFEFEFEu;
    return (((t & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | t) & 0x80808080u;
}
__device__ __forceinline__ uint32_t bytes_at_most(uint32_t x, uint32_t y) {
    const uint32_t z = (y | 0x80808080u) - (x & 0x7F7F7F7Fu);
    return ((y & ~x) | (~(x ^ y) & z)) & 0x80808080u;
}
// Codes 0..7 of 16 agents in w (byte j of word d: agent 4 d + j), those in
// valid (bit 8 j + d), counted in byte counters.
__device__ __forceinline__ void count_codes(const uint32_t (&w)[4], uint32_t valid, uint32_t& lo, uint32_t& hi) {
    uint32_t p[3];
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        p[b] = 0;
#pragma unroll
        for (int d = 0; d < 4; ++d) p[b] |= (d >= b ? w[d] << (d - b) : w[d] >> (b - d)) & (0x01010101u << d);
    }
    const uint32_t q0 = ~p[0], a = ~(p[1] | p[2]) & valid, c = p[1] & ~p[2] & valid, e = p[2] & ~p[1] & valid,
                   f = p[1] & p[2] & valid;
    lo = __popc(a & q0) | (__popc(a & p[0]) << 8) | (__popc(c & q0) << 16) | (__popc(c & p[0]) << 24);
    hi = __popc(e & q0) | (__popc(e & p[0]) << 8) | (__popc(f & q0) << 16) | (__popc(f & p[0]) << 24);
}

// One sweep block (kSweepThreads threads) over agents [t0, t0 + kSweepTile)
// of a population of N: recover (infection day <= current_day - (latent +
// infectious days), the reference's current_day - 10), count the 8 status
// codes per strain and stage the ids (+ id_bias) of infected agents.
// (kernel_countInfectedStatusAndRecover PandemicSim.cu:2097-2192,
//  daily_buildInfectedArray_global :2207-2224.)  The status arrays hold
// whole uint4 words past N.  Four agents per 32-bit operation: agent by agent
// the vector instructions, not memory, set its time (50M agents 47 us, now 35:
// 2.9 TB/s).
__device__ __forceinline__ void sweep_block(const Model& M, int64_t N, int day, int64_t t0, uint8_t* __restrict__ st_p,
                                            uint8_t* __restrict__ st_s, const uint8_t* __restrict__ dy_p,
                                            const uint8_t* __restrict__ dy_s, uint32_t* __restrict__ counts16,
                                            uint32_t* __restrict__ ninf_out, int32_t* __restrict__ stage,
                                            int32_t id_bias) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t a0 = t0 + (int64_t)tid * kSweepPer;
    static_assert(kSweepPer == 16, "four words of four agents");
    const bool full = a0 + kSweepPer <= N;
    uint32_t valid = 0x0F0F0F0Fu;
    if (!full) {
        valid = 0;
#pragma unroll
        for (int i = 0; i < kSweepPer; ++i) valid |= (a0 + i < N ? 1u : 0u) << (8 * (i % 4) + i / 4);
    }
    auto load = [&](const uint8_t* src, uint32_t (&w)[4]) {
        uint4 v = make_uint4(0, 0, 0, 0);
        if (a0 < N) v = *reinterpret_cast<const uint4*>(src + a0);
        w[0] = v.x, w[1] = v.y, w[2] = v.z, w[3] = v.w;
    };
    uint8_t* const st[2] = {st_p, st_s};
    const uint8_t* const dy[2] = {dy_p, dy_s};
    uint32_t w[2][4], inf = 0, lo[2], hi[2];
    load(st_p, w[0]);
    load(st_s, w[1]);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        uint32_t x[4], any = 0;
#pragma unroll
        for (int d = 0; d < 4; ++d) any |= x[d] = bytes_infected(w[k][d]) & (valid << (7 - d));
        const int due = day - (M.lat[k] + M.dur[k]);
        if (due >= 0 && any) {
            uint32_t v[4], rec = 0;
            load(dy[k], v);
            const uint32_t due4 = (uint32_t)min(due, 255) * 0x01010101u;
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const uint32_t m = x[d] & bytes_at_most(v[d], due4);
                rec |= m;
                w[k][d] &= ~(m | (m - (m >> 7)));
                x[d] &= ~m;
            }
            static_assert(kRecovered == 0, "recovered by clearing");
            if (rec) {
                if (full) {
                    *reinterpret_cast<uint4*>(st[k] + a0) = make_uint4(w[k][0], w[k][1], w[k][2], w[k][3]);
                } else {
                    for (int i = 0; i < kSweepPer; ++i)
                        if (a0 + i < N) st[k][a0 + i] = (uint8_t)(w[k][i / 4] >> (8 * (i % 4)));
                }
            }
        }
#pragma unroll
        for (int d = 0; d < 4; ++d) inf |= x[d] >> (7 - d);
        count_codes(w[k], valid, lo[k], hi[k]);
    }
    __shared__ uint32_t s_cnt[kSweepThreads / 64][16];
    __shared__ uint32_t s_inf[kSweepThreads / 64];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        uint32_t v[8];
        wave_sum_bins8(lo[k], hi[k], v);
        if (lane == 63) {
#pragma unroll
            for (int b = 0; b < 8; ++b) s_cnt[wave][8 * k + b] = v[b];
        }
    }
    const uint32_t ninf = (uint32_t)__popc(inf);
    const uint32_t inc = full_wave_scan(ninf);
    if (lane == 63) s_inf[wave] = inc;
    __syncthreads();
    uint32_t wbase = 0, total = 0;
#pragma unroll
    for (int i = 0; i < kSweepThreads / 64; ++i) {
        if (i < wave) wbase += s_inf[i];
        total += s_inf[i];
    }
    uint32_t pos = wbase + inc - ninf;
    // Bit 8 j + d -> 4 j + d -> 4 d + j: the agents in order.
    uint32_t m = (inf & 0xFu) | ((inf >> 4) & 0xF0u) | ((inf >> 8) & 0xF00u) | ((inf >> 12) & 0xF000u);
    uint32_t t = (m ^ (m >> 3)) & 0x0A0Au;
    m ^= t ^ (t << 3);
    t = (m ^ (m >> 6)) & 0x00CCu;
    m ^= t ^ (t << 6);
    const int32_t id0 = id_bias + (int32_t)a0;
    while (m) {
        stage[pos++] = id0 + __ffs(m) - 1;
        m &= m - 1;
    }
    if (tid < 16) {
        uint32_t s = 0;
#pragma unroll
        for (int i = 0; i < kSweepThreads / 64; ++i) s += s_cnt[i][tid];
        counts16[tid] = s;
    }
    if (tid == 0) *ninf_out = total;
}

// ---------------- errand-table selection ----------------

__device__ __forceinline__ bool is_marked(const uint32_t* __restrict__ mark, uint32_t key) {
    return (mark[key >> 5] >> (key & 31)) & 1u;
}

// One selection block (kSelThreads threads) over the agents from blk_a0 of a
// population of N: regenerates each agent's errand keys (weekday_keys or
// hour * E + location - base) and writes to sk/si, in ascending agent order,
// the pairs (kbias + key, agent) whose bucket kbias + key is marked, or every
// pair when all is set (through LDS, so the global writes are contiguous).
// Block-ordered output keeps the ids ascending within every bucket (equal
// buckets never come from two hours of one agent).  *cnt_out (if set) gets
// the number written.  Returns false if a destination fell outside the
// layout.
template <int PER, bool WEEKEND>
__device__ __forceinline__ bool select_block(const Model& M, uint64_t eoff, const uint8_t* __restrict__ age,
                                             const uint32_t* __restrict__ mark, uint32_t kbias, bool all,
                                             int64_t blk_a0, int64_t N, uint32_t* __restrict__ sk,
                                             int32_t* __restrict__ si, uint32_t* __restrict__ cnt_out) {
    constexpr int KPA = WEEKEND ? 3 : 2;  // keys per agent
    constexpr int NK = PER * KPA;
    const int64_t a0 = blk_a0 + (int64_t)threadIdx.x * PER;
    uint32_t key[NK];
    uint32_t sel = 0;
    bool bad = false;
    const ErrandWalk wk = pinned(WEEKEND ? M.we_walk : M.wd_walk);
    if (WEEKEND) {
        const int base = M.we_base, E = M.we_E;
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int64_t p = a0 + q;
            key[3 * q] = key[3 * q + 1] = key[3 * q + 2] = 0;
            if (p < N) {
                int32_t hour[3], loc[3];
                weekend_errands(M, wk, eoff + (uint64_t)(int64_t)(2 * (int32_t)p), hour, loc);
#pragma unroll
                for (int e = 0; e < 3; ++e) {
                    int32_t l = loc[e] - base;
                    if ((uint32_t)l >= (uint32_t)E) {
                        bad = true;
                        l = min(max(l, 0), E - 1);
                    }
                    const uint32_t k = kbias + (uint32_t)(hour[e] * E + l);
                    key[3 * q + e] = k;
                    if (all || is_marked(mark, k)) sel |= 1u << (3 * q + e);
                }
            }
        }
    } else {
        // The thread's ages in one load when its agents are all inside the
        // population (a0 is a multiple of PER; age is PER-byte aligned).
        uint8_t ag[PER];
        if (PER == 8 && a0 + PER <= N) {
            const uint2 v = *reinterpret_cast<const uint2*>(age + a0);
            memcpy(ag, &v, 8);
        } else {
#pragma unroll
            for (int q = 0; q < PER; ++q) ag[q] = a0 + q < N ? age[a0 + q] : 0;
        }
#pragma unroll
        for (int q = 0; q < PER / 2; ++q) {
            const int64_t g = a0 / 2 + q;
            key[4 * q] = key[4 * q + 1] = key[4 * q + 2] = key[4 * q + 3] = 0;
            if (2 * g < N) {
                const U4 u = draw4(eoff + (uint64_t)g, M.key0, M.key1);
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const int64_t p = 2 * g + k;
                    if (p < N) {
                        int32_t d1, d2;
                        weekday_dests(M, wk, u.w[2 * k], u.w[2 * k + 1], ag[2 * q + k] == kAgeAdult, d1, d2);
                        const int i = 4 * q + 2 * k;
                        bad |= !weekday_keys(M, d1, d2, key[i], key[i + 1]);
                        key[i] += kbias;
                        key[i + 1] += kbias;
                        if (all || is_marked(mark, key[i])) sel |= 1u << i;
                        if (all || is_marked(mark, key[i + 1])) sel |= 1u << (i + 1);
                    }
                }
            }
        }
    }
    // Block-wide exclusive scan of the per-thread counts.
    __shared__ uint32_t s_w[kSelThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t cnt = (uint32_t)__popc(sel);
    const uint32_t inc = wave_incl_scan(cnt, lane);
    if (lane == 63) s_w[wave] = inc;
    __syncthreads();
    uint32_t pos = 0, total = 0;
#pragma unroll
    for (int w = 0; w < kSelThreads / 64; ++w) {
        if (w < wave) pos += s_w[w];
        total += s_w[w];
    }
    pos += inc - cnt;
    // Staged at j + j / 16: dense blocks put thread t's pairs at 16t + i,
    // which the padding spreads over distinct LDS banks.
    constexpr int SN = kSelThreads * NK + kSelThreads * NK / 16;
    __shared__ uint32_t s_k[SN];
    __shared__ int32_t s_i[SN];
#pragma unroll
    for (int i = 0; i < NK; ++i)
        if (sel & (1u << i)) {
            s_k[pos + (pos >> 4)] = key[i];
            s_i[pos + (pos >> 4)] = (int32_t)(a0 + i / KPA);
            pos++;
        }
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < total; j += kSelThreads) {
        sk[j] = s_k[j + (j >> 4)];
        si[j] = s_i[j + (j >> 4)];
    }
    if (cnt_out && threadIdx.x == 0) *cnt_out = total;
    return !bad;
}

// ---------------- contacts ----------------

// device_selectRandomPersonFromLocation (PandemicSim.cu:2028-2071) with
// device_getVictimAtIndex (:2016-2025): household members are consecutive ids.
__device__ __forceinline__ int select_person(int32_t infector, int32_t loc_off, int32_t loc_count, uint32_t r,
                                             int type, const int32_t* __restrict__ people, int32_t& victim) {
    if (loc_count > 1) {
        int vo = (int)(r % (uint32_t)loc_count);
        int32_t v = (type == CT_HOME) ? loc_off + vo : people[loc_off + vo];
        if (v == infector) {
            vo = (vo + 1) % loc_count;
            v = (type == CT_HOME) ? loc_off + vo : people[loc_off + vo];
        }
        victim = v;
        return type;
    }
    victim = loc_count;
    return CT_NONE;
}

// Where the victims of an infector's contact slots come from: the household
// (slots 0..2; its members are consecutive ids), then `wpd` workplace or
// school slots, then h0 slots in the first errand location and h1 in the
// second (weekend: wpd = 0, h0 = h1 = 1), with each slot's draw (SlotDraws).  Only a
// slot whose infection draw succeeds needs its victim, so outside
// validation mode the contact kernels look victims up then (pick) instead of
// gathering one from a location table for every slot: the contact types and
// kval_sum depend on the location counts alone (select_person), and the
// victims of unsuccessful slots are never read.
// With counted tables e0off and e1off hold the errand buckets.
// (The draws are an array of their own: inside the struct they kept all of it
// in scratch memory.)
struct SlotPlan {
    int32_t hoff, hcnt, woff, wcnt, e0off, e0cnt, e1off, e1cnt;
    int wpd, h0, h1;
};
using SlotDraws = uint32_t[8];

// The victim of slot c (select_person's pick; the slot's count is > 1).
__device__ __forceinline__ int32_t pick(const SlotPlan& P, const SlotDraws& r, const int32_t* __restrict__ wp_people,
                                        const int32_t* __restrict__ er_people, int32_t infector, int c) {
    int32_t off, cnt;
    const int32_t* people;
    if (c < 3) {
        off = P.hoff;
        cnt = P.hcnt;
        people = nullptr;
    } else if (c < 3 + P.wpd) {
        off = P.woff;
        cnt = P.wcnt;
        people = wp_people;
    } else if (c < 3 + P.wpd + P.h0) {
        off = P.e0off;
        cnt = P.e0cnt;
        people = er_people;
    } else {
        off = P.e1off;
        cnt = P.e1cnt;
        people = er_people;
    }
    int32_t v;
    select_person(infector, off, cnt, r[c], people ? CT_ERRAND : CT_HOME, people, v);
    return v;
}

// The arrays of one simulation in its local numbering.  er_off is indexed by
// the simulation's bucket key; its values (and the other offsets) index the
// corresponding people arrays as given.
struct AgentArrays {
    const uint8_t* age;
    const int32_t* household;
    const int32_t* hh_off;
    const int32_t* wp_off;
    const int32_t* wp_people;
    const AgentRecord* who;
    const int32_t* er_off;
    const int32_t* er_people;
    // Counted tables (er_off, er_people unused): people per bucket, and the
    // agents' keys of the day, er_slots apart per errand.
    const uint32_t* er_cnt;
    const uint16_t* er_keys;
    int64_t er_slots;
    const uint8_t* st_p;
    const uint8_t* st_s;
    const uint8_t* dy_p;
    const uint8_t* dy_s;
    const uint8_t* gn_p;
    const uint8_t* gn_s;
    uint64_t* claim_p;
    uint64_t* claim_s;
    // Optional per-contact trace of the day (validation mode), [I * C]
    // with C = 8 weekday / 5 weekend slots per infector: victim, type, the
    // contact's location (household, workplace, location id for
    // after-school, hour * W + location for errands; also for a contact that
    // found nobody else there, whose victim is the location's count; -1 for
    // an unused or dropped slot) and the
    // attempts that succeeded on a susceptible victim (2 pandemic, 1
    // seasonal; which of them won the victim is settled after all claims).
    int32_t* trace_victim;
    uint8_t* trace_type;
    int32_t* trace_loc;
    uint8_t* trace_attempt;
    // Optional per-slot draw record (validation mode), [I * C]: trace_draw
    // bit 1 / bit 0 = the pandemic / seasonal draw y < p * kval succeeded,
    // whatever the victim's state; trace_prof = the profile each strain's
    // draw would give (device_getInfectionProfile, PandemicSim.cu:3974-3988),
    // pandemic in the low nibble, seasonal in the high nibble.  The
    // reference computes both for every slot (PandemicSim.cu:3195-3211).
    uint8_t* trace_draw;
    uint8_t* trace_prof;

    __host__ __device__ void clear_trace() {
        trace_victim = trace_loc = nullptr;
        trace_type = trace_attempt = trace_draw = trace_prof = nullptr;
    }
};

// Strain state of an infector (device_processContacts, PandemicSim.cu:3125-3175):
// profile and shedding day if infectious today, else -1.  Infectious while
// lat <= day - infection day < lat + dur (the reference: 0 <= . < 10), at
// shedding index day - infection day - lat.
struct Infectivity {
    int prof_p, dd_p, prof_s, dd_s;
    uint8_t gen_p, gen_s;
};

__device__ __forceinline__ Infectivity infectivity(const Model& M, const AgentArrays& A, int32_t idx, int day) {
    Infectivity f;
    f.prof_p = f.prof_s = -1;
    f.dd_p = f.dd_s = 0;
    f.gen_p = f.gen_s = kGenNone;
    const uint8_t sp = A.st_p[idx], ss = A.st_s[idx];
    if (sp >= kInfected) {
        const int dd = day - (int)A.dy_p[idx] - M.lat[0];
        if (dd >= 0 && dd < M.dur[0]) {
            f.prof_p = sp - kInfected;
            f.dd_p = dd;
            f.gen_p = (uint8_t)(A.gn_p[idx] + 1);
        }
    }
    if (ss >= kInfected) {
        const int dd = day - (int)A.dy_s[idx] - M.lat[1];
        if (dd >= 0 && dd < M.dur[1]) {
            f.prof_s = ss - kInfected;
            f.dd_s = dd;
            f.gen_s = (uint8_t)(A.gn_s[idx] + 1);
        }
    }
    return f;
}

// The same in 30 bits.
__device__ __forceinline__ uint32_t pack_infectivity(const Infectivity& f) {
    return (uint32_t)(f.prof_p + 1) | ((uint32_t)f.dd_p << 3) | ((uint32_t)(f.prof_s + 1) << 7) |
           ((uint32_t)f.dd_s << 10) | ((uint32_t)f.gen_p << 14) | ((uint32_t)f.gen_s << 22);
}
__device__ __forceinline__ Infectivity unpack_infectivity(uint32_t w) {
    return Infectivity{(int)(w & 7u) - 1, (int)((w >> 3) & 15u), (int)((w >> 7) & 7u) - 1, (int)((w >> 10) & 15u),
                       (uint8_t)(w >> 14), (uint8_t)(w >> 22)};
}

// Whether the infector can infect at all today: with alpha*factor <= 0 every
// draw y >= 0 fails y < p*kval, so contacts need not be generated.
__device__ __forceinline__ bool can_infect(const Model& M, const Infectivity& f) {
    const bool p = f.prof_p >= 0 && M.shed[f.prof_p][f.dd_p] * M.factor[0] > 0.f;
    const bool s = f.prof_s >= 0 && M.shed[f.prof_s][f.dd_s] * M.factor[1] > 0.f;
    return p || s;
}

// The words of an infector's success draws (4 counters; the 5 weekend slots
// reach 11 words of them): slot c uses words 2c (pandemic) and 2c + 1
// (seasonal).
struct SuccessDraws {
    uint32_t u[16];
};
template <int C>
__device__ __forceinline__ void success_draws(const Model& M, uint64_t M2, SuccessDraws& d) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        U4 w{};
        if (q < (C + 1) / 2) w = draw4(M2 + (uint64_t)q, M.key0, M.key1);
#pragma unroll
        for (int j = 0; j < 4; ++j) d.u[4 * q + j] = w.w[j];
    }
}

// Per-contact draws and claims (device_processContacts PandemicSim.cu:3177-3231).
// Every successful attempt on a victim that is susceptible at the start of
// the day posts ((pos*8 + slot) << 32 | gen << 8 | profile) with a 64-bit
// atomicMin into the victim's claim word; the first poster is told so.
// vic: the slots' victims when `resolved` (validation mode), else filled
// here for the slots whose draw succeeds (pick).
template <int C>
__device__ __forceinline__ void process_contacts(const Model& M, const AgentArrays& A, const Infectivity& f, int kval_sum,
                                                 int32_t (&vic)[8], const int (&typ)[8], const SlotPlan& P,
                                                 const SlotDraws& slot_draws, bool resolved, int32_t idx, const SuccessDraws& draws, uint32_t pos,
                                                 bool (&newp)[8], bool (&news)[8]) {
    const float prob_p = f.prof_p >= 0 ? infection_probability(M, f.prof_p, f.dd_p, 0, kval_sum) : -1.f;
    const float prob_s = f.prof_s >= 0 ? infection_probability(M, f.prof_s, f.dd_s, 1, kval_sum) : -1.f;
    const uint32_t(&u)[16] = draws.u;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const float kv = typ[c] == CT_NONE ? 0.f : 1.f;
        uint8_t attempt = 0;
        const bool draw_p = unit_float(u[2 * c]) < prob_p * kv;
        const bool draw_s = unit_float(u[2 * c + 1]) < prob_s * kv;
        int32_t v = vic[c];
        if (!resolved && (draw_p || draw_s)) {  // kv = 1: a real contact, count > 1
            v = pick(P, slot_draws, A.wp_people, A.er_people, idx, c);
            vic[c] = v;
        }
        if (A.trace_draw) {
            const int64_t e = (int64_t)pos * C + c;
            A.trace_draw[e] = (uint8_t)((draw_p ? 2 : 0) | (draw_s ? 1 : 0));
            A.trace_prof[e] = (uint8_t)(infection_profile(M, u[2 * c] ^ u[(2 * c + 1) % 16]) |
                                        (infection_profile(M, u[2 * c + 1] ^ u[(2 * c + 2) % 16]) << 4));
        }
        if (draw_p) {
            if (A.st_p[v] == kSusceptible) {
                const uint32_t prof = infection_profile(M, u[2 * c] ^ u[(2 * c + 1) % 16]);
                const uint64_t claim = ((uint64_t)(pos * 8u + (uint32_t)c) << 32) | ((uint32_t)f.gen_p << 8) | prof;
                const uint64_t old = atomicMin((unsigned long long*)&A.claim_p[v], (unsigned long long)claim);
                newp[c] = old == ~0ull;
                attempt |= 2;
            }
        }
        if (draw_s) {
            if (A.st_s[v] == kSusceptible) {
                const uint32_t prof = infection_profile(M, u[2 * c + 1] ^ u[(2 * c + 2) % 16]);
                const uint64_t claim = ((uint64_t)(pos * 8u + (uint32_t)c) << 32) | ((uint32_t)f.gen_s << 8) | prof;
                const uint64_t old = atomicMin((unsigned long long*)&A.claim_s[v], (unsigned long long)claim);
                news[c] = old == ~0ull;
                attempt |= 1;
            }
        }
        if (A.trace_attempt) A.trace_attempt[(int64_t)pos * C + c] = attempt;
    }
}

// Appends the victims each thread posted first to the claim lists (as
// id_bias + victim).  All threads of the block must call.  One atomic per
// block and strain: atomics on one address pass at about 2 ns each, so one
// per wave took longer than the contacts themselves.
__device__ __forceinline__ void append_claims(uint32_t* n_claimed, int32_t* __restrict__ list_p,
                                              int32_t* __restrict__ list_s, int32_t id_bias,
                                              const int32_t (&vic)[8], const bool (&newp)[8], const bool (&news)[8],
                                              int lane) {
    __shared__ uint32_t s_cnt[2], s_base[2];
    uint32_t n[2] = {0, 0};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        n[0] += newp[c];
        n[1] += news[c];
    }
    if (threadIdx.x < 2) s_cnt[threadIdx.x] = 0;
    __syncthreads();
    uint32_t at[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const uint32_t inc = wave_incl_scan(n[k], lane);
        const uint32_t total = __shfl(inc, 63, 64);
        uint32_t base = 0;
        if (lane == 0 && total) base = atomicAdd(&s_cnt[k], total);
        at[k] = __shfl(base, 0, 64) + inc - n[k];
    }
    __syncthreads();
    if (threadIdx.x < 2 && s_cnt[threadIdx.x])
        s_base[threadIdx.x] = atomicAdd(&n_claimed[threadIdx.x], s_cnt[threadIdx.x]);
    __syncthreads();
    uint32_t ip = s_base[0] + at[0], is = s_base[1] + at[1];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        if (newp[c]) list_p[ip++] = id_bias + vic[c];
        if (news[c]) list_s[is++] = id_bias + vic[c];
    }
}

__device__ __forceinline__ void clear_contacts(int32_t (&vic)[8], int (&typ)[8], bool (&newp)[8], bool (&news)[8]) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        vic[c] = -1;
        typ[c] = CT_NONE;
        newp[c] = news[c] = false;
    }
}

// The same with a queue (counted tables): successful slots are queued and
// claimed together by the block (PickPush), so a wave does not go through the
// look-up chain of every slot in which one of its lanes succeeds.  All
// threads of the block must call, the idle ones with active false.
template <int C, class Queue>
__device__ __forceinline__ void queue_contacts(const Model& M, bool active, const Infectivity& f, int kval_sum,
                                               const int (&typ)[8], const SlotPlan& P,
                                               const SlotDraws& slot_draws, int32_t idx, const SuccessDraws& draws,
                                               uint32_t pos, const Queue& queue) {
    float prob_p = -1.f, prob_s = -1.f;
    if (active && f.prof_p >= 0) prob_p = infection_probability(M, f.prof_p, f.dd_p, 0, kval_sum);
    if (active && f.prof_s >= 0) prob_s = infection_probability(M, f.prof_s, f.dd_s, 1, kval_sum);
    const uint32_t(&u)[16] = draws.u;
    uint32_t hit_p = 0, hit_s = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const float kv = typ[c] == CT_NONE ? 0.f : 1.f;
        hit_p |= (unit_float(u[2 * c]) < prob_p * kv ? 1u : 0u) << c;
        hit_s |= (unit_float(u[2 * c + 1]) < prob_s * kv ? 1u : 0u) << c;
    }
    const uint32_t hit = active ? hit_p | hit_s : 0u;  // kv = 1: real contacts, count > 1
    // In registers: selects between the plan's fields would become loads from
    // scratch memory.
    int32_t hoff = P.hoff, hcnt = P.hcnt, woff = P.woff, wcnt = P.wcnt, e0off = P.e0off, e0cnt = P.e0cnt,
            e1off = P.e1off, e1cnt = P.e1cnt, wpd = P.wpd, h0 = P.h0;
    asm volatile("" : "+v"(hoff), "+v"(hcnt), "+v"(woff), "+v"(wcnt), "+v"(e0off), "+v"(e0cnt), "+v"(e1off),
                 "+v"(e1cnt), "+v"(wpd), "+v"(h0));
    // All slots in one turn when the block's successes fit the queue, else
    // two slots (at most 2 per thread) per turn.
    const int step = queue.fits((uint32_t)__popc(hit)) ? C : 2;
    for (int c0 = 0; c0 < C; c0 += step) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            if (c >= c0 && c < c0 + step && ((hit >> c) & 1u)) {
                const uint32_t prof_p = infection_profile(M, u[2 * c] ^ u[(2 * c + 1) % 16]);
                const uint32_t prof_s = infection_profile(M, u[2 * c + 1] ^ u[(2 * c + 2) % 16]);
                const bool home = c < 3, work = !home && c < 3 + wpd, first = c < 3 + wpd + h0;
                const int32_t off = home ? hoff : (work ? woff : (first ? e0off : e1off));
                const int32_t cnt = home ? hcnt : (work ? wcnt : (first ? e0cnt : e1cnt));
                queue.push(off, (uint32_t)cnt, slot_draws[c] % (uint32_t)cnt, home ? 1u : (work ? 2u : 0u), idx,
                           pos * 8u + (uint32_t)c,
                           f.gen_p | ((uint32_t)f.gen_s << 8) | (prof_p << 16) | (prof_s << 20) |
                               (((hit_p >> c) & 1u) << 24) | (((hit_s >> c) & 1u) << 25));
            }
        }
        queue.flush();
    }
}

// No queue: errand victims come from the sorted table.
struct NoQueue {
    static constexpr bool counted = false;
};

// People and table position (counted tables: the bucket) of an errand bucket.
template <bool COUNTED>
__device__ __forceinline__ void errand_bucket(const AgentArrays& A, uint32_t key, int32_t& off, int32_t& cnt) {
    if (COUNTED) {
        off = (int32_t)key;
        cnt = (int32_t)A.er_cnt[key];
    } else {
        off = A.er_off[key];
        cnt = A.er_off[key + 1] - off;
    }
}

// D6w + D7: one infector of kernel_doWeekday (PandemicSim.cu:3236-3308) with
// device_makeContacts_weekday (:1669-1829).  idx: the infector; pos: its
// position in the day's infected list; cbase, eoff: the day's contact and
// errand counters.
// With a queue every thread of the block calls, the idle ones with active
// false.
template <class Queue>
__device__ __forceinline__ void weekday_contacts(const Model& M, const AgentArrays& A, bool active,
                                                 const Infectivity& f, int day, uint64_t cbase,
                                                 uint64_t eoff, int32_t idx, int64_t pos,
                                                 int32_t (&vic)[8], int (&typ)[8], bool (&newp)[8],
                                                 bool (&news)[8], const SuccessDraws& draws, const Queue& queue) {
    const bool resolved = A.trace_victim != nullptr;
    SlotPlan P{};
    SlotDraws r = {};
    int kval = 0;
    if (active) {
        if constexpr (!Queue::counted) {  // (queued infectors can)
            if (!can_infect(M, f) && !A.trace_victim) return;
        }
        const uint64_t Mc = cbase + (uint64_t)(6 * pos);
        const U4 ua = draw4(Mc, M.key0, M.key1);
        const U4 ub = draw4(Mc + 1, M.key0, M.key1);
        const uint32_t(&u)[8] = r;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            r[q] = ua.w[q];
            r[4 + q] = ub.w[q];
        }
        const AgentRecord me = A.who[idx];
        const bool adult = record_adult(me);
        const int32_t hoff = record_household(me), hcnt = record_household_size(me);
        // workplace (device_recalcWorkplace PandemicSim.cu:3872-3890)
        const int32_t wp = record_workplace(me);
        const int wpd = record_workplace_contacts(me);
        const int32_t woff = A.wp_off[wp];
        const int32_t wcnt = A.wp_off[wp + 1] - woff;
        // errands (device_recalc_weekdayErrandDests_assignProfile :3667-3705)
        const U4 ue = draw4(eoff + (uint64_t)(idx / 2), M.key0, M.key1);
        const int rs = 2 * (idx % 2);
        const ErrandWalk wk = pinned(M.wd_walk);
        int32_t d1, d2;
        weekday_dests(M, wk, word(ue, rs), word(ue, rs + 1), adult, d1, d2);
        const int prof = adult ? (int)((word(ue, rs) ^ word(ue, rs + 1)) % 3u) : 3;
        const int h0 = M.wd_assign[prof][0], h1 = M.wd_assign[prof][1];
        uint32_t k0, k1;
        weekday_keys(M, d1, d2, k0, k1);
        int32_t e0off, e0cnt, e1off, e1cnt;
        errand_bucket<Queue::counted>(A, k0, e0off, e0cnt);
        errand_bucket<Queue::counted>(A, k1, e1off, e1cnt);
        const int wtype = adult ? CT_WORKPLACE : CT_SCHOOL;
        const int etype = adult ? CT_ERRAND : CT_AFTERSCHOOL;
        P = SlotPlan{hoff, hcnt, woff, wcnt, e0off, e0cnt, e1off, e1cnt, wpd, h0, h1};
        int32_t where[8];  // the contact's location (trace only)
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            int t;
            if (resolved) {
                if (c < 3) {
                    t = select_person(idx, hoff, hcnt, u[c], CT_HOME, nullptr, vic[c]);
                    where[c] = A.household[idx];
                } else if (c < 3 + wpd) {
                    t = select_person(idx, woff, wcnt, u[c], wtype, A.wp_people, vic[c]);
                    where[c] = wp;
                } else {
                    const int e = c - 3 - wpd;
                    if (e < h0) {
                        t = select_person(idx, e0off, e0cnt, u[c], etype, A.er_people, vic[c]);
                        where[c] = d1;
                    } else if (e < h0 + h1) {
                        t = select_person(idx, e1off, e1cnt, u[c], etype, A.er_people, vic[c]);
                        where[c] = adult ? M.W + d2 : d2;
                    } else {
                        vic[c] = -1;
                        t = CT_NONE;
                        where[c] = -1;
                    }
                }
            } else {
                // select_person's type without the pick
                const int e = c - 3 - wpd;
                const int32_t cnt = c < 3 ? hcnt : (c < 3 + wpd ? wcnt : (e < h0 ? e0cnt : (e < h0 + h1 ? e1cnt : 0)));
                const int ty = c < 3 ? CT_HOME : (c < 3 + wpd ? wtype : etype);
                t = (e < h0 + h1 && cnt > 1) ? ty : CT_NONE;
            }
            typ[c] = t;
            kval += t != CT_NONE;
        }
        apply_drops(M, day, false, Mc, 8, vic, typ);
        if (A.trace_victim) {
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                A.trace_victim[pos * 8 + c] = vic[c];
                A.trace_type[pos * 8 + c] = (uint8_t)typ[c];
                A.trace_loc[pos * 8 + c] = vic[c] < 0 ? -1 : where[c];
            }
        }
    }
    // Traced days run the draws of every infector, as the reference does: an
    // infector that cannot infect has p <= 0 (or NaN), so none of its draws
    // succeeds and it posts no claim.
    if constexpr (Queue::counted)
        queue_contacts<8>(M, active, f, kval, typ, P, r, idx, draws, (uint32_t)pos, queue);
    else if (can_infect(M, f) || A.trace_draw)
        process_contacts<8>(M, A, f, kval, vic, typ, P, r, resolved, idx, draws, (uint32_t)pos, newp, news);
    else if (A.trace_attempt)
        for (int c = 0; c < 8; ++c) A.trace_attempt[pos * 8 + c] = 0;
}

// D6e + D7: one infector of kernel_doWeekend (PandemicSim.cu:3311-3379) with
// device_makeContacts_weekend (:1833-1950).
template <class Queue>
__device__ __forceinline__ void weekend_contacts(const Model& M, const AgentArrays& A, bool active,
                                                 const Infectivity& f, int day, uint64_t cbase,
                                                 uint64_t eoff, int32_t idx, int64_t pos, int32_t (&vic)[8],
                                                 int (&typ)[8], bool (&newp)[8], bool (&news)[8],
                                                 const SuccessDraws& draws, const Queue& queue) {
    const bool resolved = A.trace_victim != nullptr;
    SlotPlan P{};
    SlotDraws r = {};
    int kval = 0;
    if (active) {
        if constexpr (!Queue::counted) {
            if (!can_infect(M, f) && !A.trace_victim) return;
        }
        const uint64_t Mc = cbase + (uint64_t)(6 * pos);
        const U4 u = draw4(Mc, M.key0, M.key1);
        const AgentRecord me = A.who[idx];
        const int32_t hoff = record_household(me), hcnt = record_household_size(me);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            if (resolved)
                typ[c] = select_person(idx, hoff, hcnt, u.w[c], CT_HOME, nullptr, vic[c]);
            else
                typ[c] = hcnt > 1 ? CT_HOME : CT_NONE;
        }
        const int prof = (int)(u.w[3] % 6u);
        uint32_t v32[2];
        draw2x32((uint32_t)(Mc + 1), (uint32_t)M.key0, (uint32_t)M.key1, v32);
        const int32_t hh = resolved ? A.household[idx] : 0;
        int32_t where[5] = {hh, hh, hh, -1, -1};  // the contact's location (trace only)
        int32_t eo[2], ec[2];
        if (Queue::counted && A.er_keys) {
            const uint16_t* keys = A.er_keys + idx;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                errand_bucket<Queue::counted>(A, keys[M.we_assign[prof][k] * A.er_slots], eo[k], ec[k]);
                typ[3 + k] = ec[k] > 1 ? CT_ERRAND : CT_NONE;
            }
        } else {
            const ErrandWalk wk = pinned(M.we_walk);
            int32_t hour[3], loc[3];
            weekend_errands(M, wk, eoff + (uint64_t)(int64_t)(2 * idx), hour, loc);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int slot = M.we_assign[prof][k];
                const int hsel = slot == 0 ? hour[0] : (slot == 1 ? hour[1] : hour[2]);
                const int lsel = slot == 0 ? loc[0] : (slot == 1 ? loc[1] : loc[2]);
                const int32_t l = min(max(lsel - M.we_base, 0), M.we_E - 1);
                const int32_t key = hsel * M.we_E + l;
                errand_bucket<Queue::counted>(A, (uint32_t)key, eo[k], ec[k]);
                if (resolved)
                    typ[3 + k] = select_person(idx, eo[k], ec[k], v32[k], CT_ERRAND, A.er_people, vic[3 + k]);
                else
                    typ[3 + k] = ec[k] > 1 ? CT_ERRAND : CT_NONE;
                where[3 + k] = hsel * M.W + lsel;
            }
        }
        P = SlotPlan{hoff, hcnt, 0, 0, eo[0], ec[0], eo[1], ec[1], 0, 1, 1};
#pragma unroll
        for (int q = 0; q < 3; ++q) r[q] = u.w[q];
        r[3] = v32[0];
        r[4] = v32[1];
#pragma unroll
        for (int c = 0; c < 5; ++c) kval += typ[c] != CT_NONE;
        apply_drops(M, day, true, Mc, 5, vic, typ);
        if (A.trace_victim) {
#pragma unroll
            for (int c = 0; c < 5; ++c) {
                A.trace_victim[pos * 5 + c] = vic[c];
                A.trace_type[pos * 5 + c] = (uint8_t)typ[c];
                A.trace_loc[pos * 5 + c] = vic[c] < 0 ? -1 : where[c];
            }
        }
    }
    // Traced days run the draws of every infector, as the reference does: an
    // infector that cannot infect has p <= 0 (or NaN), so none of its draws
    // succeeds and it posts no claim.
    if constexpr (Queue::counted)
        queue_contacts<5>(M, active, f, kval, typ, P, r, idx, draws, (uint32_t)pos, queue);
    else if (can_infect(M, f) || A.trace_draw)
        process_contacts<5>(M, A, f, kval, vic, typ, P, r, resolved, idx, draws, (uint32_t)pos, newp, news);
    else if (A.trace_attempt)
        for (int c = 0; c < 5; ++c) A.trace_attempt[pos * 5 + c] = 0;
}

// Whether any contact draw of an infector can succeed: y < p for one of its
// slots' uniforms against the p that a contact count of at least kval gives
// (the rounded quotient only falls with the count).  With kval = 1 it needs
// nothing but the infector's strain state and its own draws.
template <int C>
__device__ __forceinline__ bool may_infect(const Model& M, const Infectivity& f, const SuccessDraws& d, int kval) {
    const float bp = f.prof_p >= 0 ? infection_probability(M, f.prof_p, f.dd_p, 0, kval) : -1.f;
    const float bs = f.prof_s >= 0 ? infection_probability(M, f.prof_s, f.dd_s, 1, kval) : -1.f;
    bool any = false;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        any |= unit_float(d.u[2 * c]) < bp;
        any |= unit_float(d.u[2 * c + 1]) < bs;
    }
    return any;
}

// Contacts of the day's I infectors in two phases.  Most infectors cannot
// infect anyone today (half of the infectious days shed below 0.1%), and a
// wave holds a random mix, so instead of branching per lane a block tests T
// infectors at a time (test(pos, item, draws) -> may_infect) and queues the
// ones left, with their draws, in LDS; whenever T are queued it runs them
// together (run(active, item, draws), called by all threads).  Claims resolve by position and slot, so
// the order does not matter.  VALU bound (8 draws of ~145 instructions per
// infector before, 4 plus 8 per one left now): 50M agents x 100 days,
// contacts 41.6 -> 20.1 ms.
struct QueuedInfector {
    int32_t idx, pos, r;
};

template <int T, int C, class Test, class Run>
__device__ __forceinline__ void filtered_contacts(int64_t I, Test test, Run run) {
    constexpr int NW = 4 * ((C + 1) / 2);  // words drawn
    __shared__ QueuedInfector s_q[2 * T];
    __shared__ uint32_t s_u[NW][2 * T];
    __shared__ uint32_t s_n;
    const int tid = threadIdx.x, lane = tid & 63;
    if (tid == 0) s_n = 0;
    __syncthreads();
    const int64_t stride = (int64_t)gridDim.x * T;
    for (int64_t b0 = (int64_t)blockIdx.x * T;; b0 += stride) {
        const bool more = b0 < I;  // the last turn only empties the queue
        QueuedInfector item{};
        SuccessDraws draws{};
        if (more) {
            const int64_t pos = b0 + tid;
            const bool keep = pos < I && test(pos, item, draws);
            const uint64_t m = __ballot(keep);
            uint32_t at = 0;
            if (lane == 0 && m) at = atomicAdd(&s_n, (uint32_t)__popcll(m));
            at = __shfl(at, 0, 64);
            if (keep) {
                at += (uint32_t)__popcll(m & ((1ull << lane) - 1));
                s_q[at] = item;
#pragma unroll
                for (int j = 0; j < NW; ++j) s_u[j][at] = draws.u[j];
            }
            __syncthreads();
        }
        const uint32_t n = s_n;  // below 2T; below T on the last turn
        const uint32_t take = min(n, (uint32_t)T);
        if (take == (uint32_t)T || (!more && take)) {
            const bool active = (uint32_t)tid < take;
            if (active) {
                item = s_q[n - take + tid];
#pragma unroll
                for (int j = 0; j < NW; ++j) draws.u[j] = s_u[j][n - take + tid];
            }
            __syncthreads();
            if (tid == 0) s_n = n - take;
            run(active, item, draws);
        }
        if (!more) break;
        __syncthreads();
    }
}

// ---------------- queried-bucket marks ----------------

// Sets bit kbias + key when key < K.
__device__ __forceinline__ void set_mark(uint32_t* __restrict__ mark, int32_t key, int32_t K, uint32_t kbias) {
    if ((uint32_t)key >= (uint32_t)K) return;
    const uint32_t k = kbias + (uint32_t)key;
    const uint32_t bit = 1u << (k & 31);
    if (!(__hip_atomic_load(&mark[k >> 5], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit))
        atomicOr(&mark[k >> 5], bit);
}

// The weekday errand buckets an infector draws contacts from: hour h is
// used iff the errand profile asks for contacts in it (the workplace takes at
// most 3 of the 5 non-household slots, so the first requested hour always
// gets one; PandemicSim.cu:1776-1813).
__device__ __forceinline__ void mark_weekday(const Model& M, const AgentArrays& A, int day, uint64_t eoff, int32_t idx,
                                             uint32_t* __restrict__ mark, uint32_t kbias) {
    // The contact kernels also draw for infectors that cannot infect when
    // tracing (their contacts are traced), so their buckets are queried too.
    const Infectivity f = infectivity(M, A, idx, day);
    if (!can_infect(M, f) && !A.trace_victim) return;
    const bool adult = A.age[idx] == kAgeAdult;
    const U4 ue = draw4(eoff + (uint64_t)(idx / 2), M.key0, M.key1);
    const int rs = 2 * (idx % 2);
    const ErrandWalk wk = pinned(M.wd_walk);
    int32_t d1, d2;
    weekday_dests(M, wk, word(ue, rs), word(ue, rs + 1), adult, d1, d2);
    uint32_t k0, k1;
    weekday_keys(M, d1, d2, k0, k1);
    const int prof = adult ? (int)((word(ue, rs) ^ word(ue, rs + 1)) % 3u) : 3;
    if (M.wd_assign[prof][0] > 0) set_mark(mark, (int32_t)k0, M.wd_K, kbias);
    if (M.wd_assign[prof][1] > 0) set_mark(mark, (int32_t)k1, M.wd_K, kbias);
}

// The two weekend errand buckets of an infector (PandemicSim.cu:1891-1946).
__device__ __forceinline__ void mark_weekend(const Model& M, const AgentArrays& A, int day, uint64_t cbase,
                                             uint64_t eoff, int64_t pos, int32_t idx, uint32_t* __restrict__ mark,
                                             uint32_t kbias) {
    const Infectivity f = infectivity(M, A, idx, day);
    if (!can_infect(M, f) && !A.trace_victim) return;  // as mark_weekday
    const U4 u = draw4(cbase + (uint64_t)(6 * pos), M.key0, M.key1);
    const int prof = (int)(u.w[3] % 6u);
    const ErrandWalk wk = pinned(M.we_walk);
    int32_t hour[3], loc[3];
    weekend_errands(M, wk, eoff + (uint64_t)(int64_t)(2 * idx), hour, loc);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int slot = M.we_assign[prof][k];
        const int hsel = slot == 0 ? hour[0] : (slot == 1 ? hour[1] : hour[2]);
        const int lsel = slot == 0 ? loc[0] : (slot == 1 ? loc[1] : loc[2]);
        set_mark(mark, hsel * M.we_E + (lsel - M.we_base), kWeHours * M.we_E, kbias);
    }
}

// ---------------- kernels used by both engines ----------------
// (internal linkage: each translation unit compiles its own copy)
namespace {

// Compaction of per-block staged runs (counts cnt, offsets off) into one list.
__global__ void k_compact_runs(const int32_t* __restrict__ skip, const uint32_t* __restrict__ stage_keys,
                               const int32_t* __restrict__ stage_ids, const uint32_t* __restrict__ blk_cnt,
                               const uint32_t* __restrict__ blk_off, uint32_t* __restrict__ sel_keys,
                               int32_t* __restrict__ sel_ids, int stage_stride, uint32_t* __restrict__ n_sel,
                               int nblk) {
    if (*skip) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) *n_sel = blk_off[nblk - 1] + blk_cnt[nblk - 1];
    const uint32_t n = blk_cnt[blockIdx.x];
    const uint32_t off = blk_off[blockIdx.x];
    const int64_t src = (int64_t)blockIdx.x * stage_stride;
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
        sel_keys[off + i] = stage_keys[src + i];
        sel_ids[off + i] = stage_ids[src + i];
    }
}

// Winners write status = profile, day = current_day + 1, generation
// (device_setInfectionStatus PandemicSim.cu:3048-3067); claim words reset.
__device__ __forceinline__ void apply_claims(const DayState* st, uint64_t* __restrict__ claim_p,
                        uint64_t* __restrict__ claim_s, const int32_t* __restrict__ list_p,
                        const int32_t* __restrict__ list_s, uint8_t* __restrict__ st_p, uint8_t* __restrict__ st_s,
                        uint8_t* __restrict__ dy_p, uint8_t* __restrict__ dy_s, uint8_t* __restrict__ gn_p,
                        uint8_t* __restrict__ gn_s) {
    const uint32_t np = st->n_claimed[0], ns = st->n_claimed[1];
    const uint8_t dset = (uint8_t)(st->day + 1);
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < (int64_t)np + ns; i += stride) {
        if (i < np) {
            const int32_t v = list_p[i];
            const uint64_t c = claim_p[v];
            st_p[v] = (uint8_t)(c & 0xFF);
            dy_p[v] = dset;
            gn_p[v] = (uint8_t)((c >> 8) & 0xFF);
            claim_p[v] = ~0ull;
        } else {
            const int32_t v = list_s[i - np];
            const uint64_t c = claim_s[v];
            st_s[v] = (uint8_t)(c & 0xFF);
            dy_s[v] = dset;
            gn_s[v] = (uint8_t)((c >> 8) & 0xFF);
            claim_s[v] = ~0ull;
        }
    }
}

__global__ void k_apply(const DayState* __restrict__ st, uint64_t* __restrict__ claim_p,
                        uint64_t* __restrict__ claim_s, const int32_t* __restrict__ list_p,
                        const int32_t* __restrict__ list_s, uint8_t* __restrict__ st_p, uint8_t* __restrict__ st_s,
                        uint8_t* __restrict__ dy_p, uint8_t* __restrict__ dy_s, uint8_t* __restrict__ gn_p,
                        uint8_t* __restrict__ gn_s) {
    if (st->done) return;
    apply_claims(st, claim_p, claim_s, list_p, list_s, st_p, st_s, dy_p, dy_s, gn_p, gn_s);
}

// Plain copy of n16 16-byte words (snapshot / restore of the agent state).
__global__ void k_copy16(const uint4* __restrict__ src, uint4* __restrict__ dst, int64_t n16) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride) dst[i] = src[i];
}

// setup_initialInfected (PandemicSim.cu:708-758).
__global__ void k_seed_infections(const int32_t* __restrict__ ids, int n_p, int n_s, uint8_t* st_p, uint8_t* st_s,
                                  uint8_t* dy_p, uint8_t* dy_s, uint8_t* gn_p, uint8_t* gn_s) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_p + n_s) return;
    const int id = ids[i];
    if (i < n_p) {
        st_p[id] = kInfected;
        dy_p[id] = 0;
        gn_p[id] = 0;
    } else {
        st_s[id] = kInfected;
        dy_s[id] = 0;
        gn_s[id] = 0;
    }
}

// Generation histograms (final_countReproduction, PandemicSim.cu:2236-2260).
__global__ void k_gen_hist(const uint8_t* __restrict__ gn_p, const uint8_t* __restrict__ gn_s, int64_t N,
                           unsigned long long* __restrict__ hist) {
    __shared__ uint32_t s_h[512];
    for (int i = threadIdx.x; i < 512; i += blockDim.x) s_h[i] = 0;
    __syncthreads();
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += stride) {
        atomicAdd(&s_h[gn_p[i]], 1u);
        atomicAdd(&s_h[256 + gn_s[i]], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 512; i += blockDim.x)
        if (s_h[i]) atomicAdd(&hist[i], (unsigned long long)s_h[i]);
}

}  // namespace
}  // namespace pt
