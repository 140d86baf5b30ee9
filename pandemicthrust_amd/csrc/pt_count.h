// pt_count.h — counted errand tables: the day's errand contacts without a
// sorted table.
//
// A contact at an errand location needs the number of people in its bucket
// (hour, location), and, only when its infection draw succeeds, the person at
// one rank of the bucket's ascending ids (select_person).  Sorting every
// (bucket, id) pair of the day to serve those few look-ups moves each pair
// two or three times through HBM.  Here the pairs are never moved:
//
//   k_count       a block per chunk of consecutive agents draws their
//                 errands, counts them per bucket in LDS and writes the
//                 counts (one matrix row per chunk) and the 2-byte keys
//   k_count_scan  per bucket, the exclusive prefix over the chunks and the
//                 total: pre[b][c] people of bucket b lie in chunks before
//                 c.  Transposed, so that a rank's chunk is found within one
//                 or two cache lines of its bucket
//   test          the day's infectors whose success draws cannot all fail
//                 (may_infect) go to a list
//   contacts      of the listed infectors, with the totals; a successful
//                 errand draw queues the pick (bucket, rank), finds the chunk
//                 holding that rank from the prefixes and marks (chunk, bucket)
//   k_collect     chunks with marks go through their keys again and list the
//                 ids of the marked buckets (about 8 per bucket and chunk)
//   k_resolve     16 lanes per pick find the id with the pick's rank within
//                 its list and post the infection claim
//
// While chunks are small (a simulation of up to a million agents), k_resolve
// looks through the chunk's keys itself, and nothing is marked or listed.
//
// A chunk's list order does not matter (ranks are taken by value), so the
// result is the id the sorted table holds at that position.
//
// Layouts of at most kCountMaxK buckets count in one block per chunk (32-bit
// counters in one CU's 160 KB LDS).  Larger ones are split into column
// groups (an hour, or kCountMaxK locations of one): k_keys_* write the keys
// by hour or group first, then k_count_group counts (chunk, group) from them,
// and k_collect_group lists; the rest is shared.
//
// Whole workloads, sorted tables before: 2.35M agents x 100 days 20.7 -> 8.9
// ms, 50M x 100 days (split) 161-175 -> 76-82 ms, 24M with 10x the locations
// (split, few infected, so only queried buckets were sorted) 35 -> 24 ms, 48
// replicates of 50k to 2M 259 -> 74 ms.
//
// Citations are relative to PandemicThrust/PandemicThrust/ of the reference.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "pt_day.h"

namespace pt {

constexpr int kCountMaxK = 40000;       // 32-bit counters: 160,000 of the 163,840 bytes of LDS
constexpr uint32_t kNoKey = 0xFFFFu;    // no pair (weekday hour 1 of a child)
constexpr int kCountMinChunk = 1024;    // agents
constexpr int kCountMaxRanges = 8;      // groups per hour: passes over its keys
constexpr int kCountMaxLen = 64;        // people per bucket of a smallest chunk (CountPlan::build)
constexpr int64_t kCountSmall = 1000000;  // agents up to which the lists' length does not matter

// One simulation's counted table in one layout (weekday or weekend).
struct CountRep {
    int64_t abase;  // first agent slot
    int64_t mbase;  // first entry of its matrices: C x K counts, K x (C + 1) prefixes
    int64_t tbase;  // first of its K totals
    int64_t qbase;  // first word of its C x qw mark words
    int32_t K, C, A, qw;  // buckets, chunks, agents per chunk, mark words per chunk
    int32_t chunk0; // first chunk (k_count block)
    // Column groups: buckets [0, E) are the first hour's, the next E (weekday:
    // the rest) the second's ...; `ranges` groups of W buckets per hour, G in
    // all (1: not split).
    int32_t E, W, ranges, G;
    int32_t toff;  // tile_off entries per tile (group lists): G + 1 and some
};

struct CountBlock {
    int32_t r, at;  // simulation; chunk (k_count, k_collect) or first bucket (k_count_scan)
};

// A successful contact draw.  Errands (kind 0): the person at `rank` of
// bucket `at`, or the next one if that is the infector itself
// (select_person).  Home (1): person `at`.  Workplace (2): the person at
// position `at` of the workplace table, or at position `rank` instead.
struct Pick {
    uint32_t at, rank;
    int32_t idx, r;      // infector, simulation
    uint32_t claim;      // position * 8 + slot
    uint32_t payload;    // gen_p | gen_s << 8 | prof_p << 16 | prof_s << 20 | draw_p << 24 | draw_s << 25 | kind << 26
};

// What contact claims are made on (agent slots of all simulations).
struct ClaimArrays {
    const uint8_t *st_p, *st_s;
    const int32_t* wp_people;
    uint64_t *claim_p, *claim_s;
    int32_t *list_p, *list_s;
    uint32_t* n_claimed;
};

// Device buffers of one layout.
struct CountTable {
    const CountRep* reps;
    const CountBlock* chunks;
    const CountBlock* scans;  // (null: one simulation, blocks in order)
    uint16_t* keys;        // keys per agent x slots (split weekday layouts: within the hour)
    int64_t slots;
    int32_t direct;        // picks are found in the keys (planes of keys per agent), without lists
    int32_t n_agents;      // direct: the simulation's agents, and its weekday buckets of hour 0
    uint32_t hour1;
    uint32_t* keys32;      // or the pairs by tile and group
    uint16_t* tile_off;    // where each tile's groups begin
    uint32_t* cnt;         // the count matrices; then, per marked (chunk, bucket), its list's position
    uint32_t* pre;         // the prefixes
    uint32_t* total;       // people per bucket
    uint32_t* marks;       // mark words
    int64_t mark_words;
    int32_t* chunk_day;    // day + 1 on which the (chunk, group) was last marked
    int32_t* list;         // ids of the marked buckets, kpa * agents per chunk
    uint32_t* n;           // [0] picks queued, [1] infectors listed, [2] list entries (split layouts), [3] k_apply_end
    // Listed infectors: agent, position, pack_infectivity, simulation (batch).
    int32_t *sv_idx, *sv_pos;
    uint32_t* sv_f;
    int32_t* sv_r;
    int32_t* lone_day;       // per simulation: day + 1 on which some bucket had a single person
    const int32_t* wp_lone;  // per simulation: some workplace has
    uint32_t *pk_bucket, *pk_want, *pk_claim, *pk_payload;  // queued picks: rank `want` of
    int32_t *pk_idx, *pk_r, *pk_chunk, *pk_len;             // the len ids of (chunk, bucket)
};

__host__ __device__ inline ClaimArrays claim_arrays(const AgentArrays& A, int32_t* list_p, int32_t* list_s,
                                                    uint32_t* n_claimed) {
    return ClaimArrays{A.st_p, A.st_s, A.wp_people, A.claim_p, A.claim_s, list_p, list_s, n_claimed};
}

// LDS queue of a contact block's successful draws: three per infector, or the
// two a turn of two slots can add (queue_contacts).
constexpr int kPickQueue = 3 * kContactThreads;
struct PickQueue {
    uint32_t n, errands, taken, base, sum, list, list_base;
    uint32_t n_claim[2], claim_base[2];
    Pick at[kPickQueue];
    int32_t claimed[2][kPickQueue];
    __device__ __forceinline__ void reset() { n = errands = taken = list = n_claim[0] = n_claim[1] = 0; }
};

// Prefixes of bucket b.
__device__ __forceinline__ const uint32_t* count_column(const CountTable& T, const CountRep& c, uint32_t b) {
    return T.pre + c.mbase + (int64_t)b * (c.C + 1);
}

// The chunk holding rank j of bucket b: the last c with pre[c][b] <= j
// (chunks without people of b share their successor's prefix).  People are
// spread evenly over the chunks, so the chunk is within C / (2 sqrt(total))
// (1 to 2) of j C / total: the eight prefixes around it nearly always hold
// it, else the window moves on.
__device__ __forceinline__ int chunk_of(const CountTable& T, const CountRep& c, uint32_t b, uint32_t j, uint32_t total,
                                        uint32_t& before, uint32_t& len) {
    constexpr int W = 8;
    const uint32_t* col = count_column(T, c, b);
    int w = (int)((float)j * (float)c.C / (float)total) - W / 2 + 1;
    for (;;) {
        w = max(0, min(w, c.C - W + 1));  // rows w .. w + W - 1 of the C + 1 (row C: the total)
        uint32_t p[W];
#pragma unroll
        for (int i = 0; i < W; ++i) p[i] = col[min(w + i, c.C)];
        if (w > 0 && j < p[0]) {
            w -= W - 1;
            continue;
        }
        if (j >= p[W - 1]) {
            w += W - 1;
            continue;
        }
        int k = 0;
#pragma unroll
        for (int i = 1; i < W; ++i)
            if (p[i] <= j) k = i;
        before = p[0];
        uint32_t next = p[1];
#pragma unroll
        for (int i = 1; i < W - 1; ++i)
            if (k == i) {
                before = p[i];
                next = p[i + 1];
            }
        len = next - before;
        return w + k;
    }
}

// Marks (chunk, bucket) for collection; true for its first mark of the day.
// (Only split layouts use the answer: without it nothing waits.)
__device__ __forceinline__ bool mark_chunk(const CountTable& T, const CountRep& c, int chunk, uint32_t b,
                                           int32_t stamp) {
    const uint32_t bit = 1u << (b & 31);
    uint32_t* word = T.marks + c.qbase + (int64_t)chunk * c.qw + (b >> 5);
    bool first = false;
    if (c.G > 1)
        first = !(atomicOr(word, bit) & bit);
    else
        atomicOr(word, bit);
    int g = 0;
    if (c.G > 1) {
        const uint32_t hour = c.G == 2 * c.ranges ? (b >= (uint32_t)c.E ? 1u : 0u) : b / (uint32_t)c.E;
        g = (int)(hour * c.ranges + (b - hour * c.E) / (uint32_t)c.W);
    }
    // (Stores to these few lines from every CU would queue up: look first.)
    int32_t* day = T.chunk_day + c.chunk0 + chunk * c.G + g;
    if (*day != stamp) *day = stamp;
    return first;
}

// Where a pick's first marks go (split layouts; n of them).
struct NewLists {
    int n;
    int64_t at[2];     // entries of the count matrix
    uint32_t len[2];
};

// A queued pick: finds and marks its chunk (and the next rank's, should the
// infector itself sit at this rank: only possible in its own chunk) and
// stores the pick as the day's i-th.
__device__ __forceinline__ void locate_pick(const CountTable& T, const Pick& p, uint32_t i, int day, NewLists& lists) {
    const CountRep c = T.reps[p.r];
    const uint32_t total = T.total[c.tbase + p.at];
    uint32_t before, len;
    const int chunk = chunk_of(T, c, p.at, p.rank, total, before, len);
    auto mark = [&](int k) {
        if (!mark_chunk(T, c, k, p.at, day + 1)) return;
        if (lists.n == 0) {
            lists.at[0] = c.mbase + (int64_t)k * c.K + p.at;
            lists.len[0] = len;
        } else {
            lists.at[1] = c.mbase + (int64_t)k * c.K + p.at;
            lists.len[1] = len;
        }
        ++lists.n;
    };
    if (!T.direct) mark(chunk);
    T.pk_bucket[i] = p.at;
    T.pk_want[i] = p.rank - before;
    T.pk_claim[i] = p.claim;
    T.pk_payload[i] = p.payload;
    T.pk_idx[i] = p.idx;
    T.pk_r[i] = p.r;
    T.pk_chunk[i] = chunk;
    T.pk_len[i] = (int32_t)len;
    if (!T.direct && chunk == p.idx / c.A) {
        const uint32_t next = p.rank + 1 == total ? 0u : p.rank + 1;
        if (next < before || next >= before + len) mark(chunk_of(T, c, p.at, next, total, before, len));
    }
}

// Posts a successful draw's claims on the person at `slot` (process_contacts);
// newp / news: first to claim that strain today.
__device__ __forceinline__ void post_claims(const ClaimArrays& C, int64_t slot, uint32_t claim, uint32_t payload,
                                            bool& newp, bool& news) {
    const uint64_t key = (uint64_t)claim << 32;
    const bool p = ((payload >> 24) & 1u) && C.st_p[slot] == kSusceptible;
    const bool s = ((payload >> 25) & 1u) && C.st_s[slot] == kSusceptible;
    if (p)
        newp = atomicMin((unsigned long long*)&C.claim_p[slot],
                         (unsigned long long)(key | ((payload & 0xFFu) << 8) | ((payload >> 16) & 0xFu))) == ~0ull;
    if (s)
        news = atomicMin((unsigned long long*)&C.claim_s[slot],
                         (unsigned long long)(key | (payload & 0xFF00u) | ((payload >> 20) & 0xFu))) == ~0ull;
}

// Every thread of the block: claims the queued home and workplace picks,
// locates the errand picks, and empties the queue.
__device__ __forceinline__ void flush_picks(const CountTable& T, const ClaimArrays& C, PickQueue& q,
                                            const DayState* __restrict__ sts) {
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t n = q.n;
    if (tid == 0 && q.errands) q.base = atomicAdd(T.n, q.errands);
    __syncthreads();
    constexpr int kTurns = kPickQueue / kContactThreads;
    NewLists lists[kTurns];
    uint32_t list_at[kTurns];
#pragma unroll
    for (int t = 0; t < kTurns; ++t) {
        const uint32_t i = (uint32_t)(t * kContactThreads + tid);
        bool newp = false, news = false;
        int64_t slot = 0;
        lists[t].n = 0;
        if (i < n) {
            const Pick p = q.at[i];
            const uint32_t kind = p.payload >> 26;
            if (kind == 0) {
                locate_pick(T, p, q.base + atomicAdd(&q.taken, 1u), sts[p.r].day, lists[t]);
                if (lists[t].n)
                    list_at[t] = atomicAdd(&q.list, lists[t].len[0] + (lists[t].n > 1 ? lists[t].len[1] : 0u));
            } else {
                const int64_t a = T.reps[p.r].abase;
                int32_t v = (int32_t)p.at;
                if (kind == 2) {
                    v = C.wp_people[a + v];
                    if (v == p.idx) v = C.wp_people[a + (int32_t)p.rank];
                }
                slot = a + v;
                post_claims(C, slot, p.claim, p.payload, newp, news);
            }
        }
        const uint64_t m[2] = {__ballot(newp), __ballot(news)};
        uint32_t at = 0;
        if (lane < 2) {
            const uint32_t k = (uint32_t)__popcll(lane ? m[1] : m[0]);
            if (k) at = atomicAdd(&q.n_claim[lane], k);
        }
        const uint64_t below = (1ull << lane) - 1;
        const uint32_t ap = __shfl(at, 0, 64), as = __shfl(at, 1, 64);
        if (newp) q.claimed[0][ap + (uint32_t)__popcll(m[0] & below)] = (int32_t)slot;
        if (news) q.claimed[1][as + (uint32_t)__popcll(m[1] & below)] = (int32_t)slot;
    }
    __syncthreads();
    if (tid < 2 && q.n_claim[tid]) q.claim_base[tid] = atomicAdd(&C.n_claimed[tid], q.n_claim[tid]);
    if (tid == 2 && q.list) q.list_base = atomicAdd(&T.n[2], q.list);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < kTurns; ++t) {
        if (lists[t].n) {
            const uint32_t start = q.list_base + list_at[t];
            T.cnt[lists[t].at[0]] = start;
            if (lists[t].n > 1) T.cnt[lists[t].at[1]] = start + lists[t].len[0];
        }
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        int32_t* list = k ? C.list_s : C.list_p;
        for (uint32_t i = tid; i < q.n_claim[k]; i += blockDim.x) list[q.claim_base[k] + i] = q.claimed[k][i];
    }
    __syncthreads();
    if (tid == 0) q.reset();
    __syncthreads();
}

// The contact kernels' queue (queue_contacts).
struct PickPush {
    static constexpr bool counted = true;
    const CountTable& T;
    const ClaimArrays& C;
    const DayState* sts;
    PickQueue* q;
    int32_t r;
    __device__ __forceinline__ void push(int32_t off, uint32_t cnt, uint32_t rank, uint32_t kind, int32_t idx,
                                         uint32_t claim, uint32_t payload) const {
        const uint32_t next = rank + 1 == cnt ? 0u : rank + 1;
        uint32_t at = (uint32_t)off;  // errand: the bucket
        if (kind == 1) {              // home: consecutive ids
            at += rank;
            if ((int32_t)at == idx) at = (uint32_t)off + next;
        } else if (kind == 2) {       // workplace: table positions
            at += rank;
            rank = (uint32_t)off + next;
        } else {
            atomicAdd(&q->errands, 1u);
        }
        q->at[atomicAdd(&q->n, 1u)] = Pick{at, rank, idx, r, claim, payload | (kind << 26)};
    }
    // Whether the block's successes (mine: this thread's) fit the queue.
    __device__ __forceinline__ bool fits(uint32_t mine) const {
        const uint32_t sum = wave_sum(mine);
        if (threadIdx.x == 0) q->sum = 0;
        __syncthreads();
        if ((threadIdx.x & 63) == 0 && sum) atomicAdd(&q->sum, sum);
        __syncthreads();
        return q->sum <= (uint32_t)kPickQueue;
    }
    __device__ __forceinline__ void flush() const {
        __syncthreads();
        if (q->n) flush_picks(T, C, *q, sts);
    }
};

namespace {

// Counting keys of two neighbouring agents (the second only if `two`) from
// their destinations; false if one lies outside its hour, which no model
// allows.  (A key below K is not enough: past its hour's end a destination has
// a bucket of the next hour.)
struct WeekdayHours {
    int32_t base0, base1;  // first location of each hour
    uint32_t E0, E1;       // locations; hour 1's buckets follow hour 0's
};
__host__ __device__ inline bool weekday_pair_keys(const WeekdayHours& H, const int32_t (&d1)[2], const int32_t (&d2)[2],
                                                  const bool (&adult)[2], bool two, uint32_t (&k0)[2],
                                                  uint32_t (&k1)[2]) {
    uint32_t top0 = 0, top1 = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const bool there = i == 0 || two;
        const uint32_t l0 = (uint32_t)(d1[i] - H.base0), l1 = (uint32_t)(d2[i] - H.base1);
        const uint32_t c0 = there ? l0 : 0u, c1 = adult[i] ? l1 : 0u;
        top0 = c0 > top0 ? c0 : top0;
        top1 = c1 > top1 ? c1 : top1;
        k0[i] = there ? l0 : kNoKey;
        k1[i] = adult[i] ? H.E0 + l1 : kNoKey;
    }
    return (top0 < H.E0) & (top1 < H.E1);
}
__host__ __device__ inline bool weekend_pair_keys(int32_t base, uint32_t E, const int32_t (&hour)[2][3],
                                                  const int32_t (&loc)[2][3], bool two, uint32_t (&k)[2][3]) {
    uint32_t top = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            const uint32_t l = (uint32_t)(loc[i][e] - base), c = i == 0 || two ? l : 0u;
            top = c > top ? c : top;
            // (hours below 10, E below 2^24: a 24-bit product)
            k[i][e] = (((uint32_t)hour[i][e] & 0xFFFFFFu) * (E & 0xFFFFFFu)) + l;
        }
    }
    return top < E;
}

// Keys and counts of a chunk.  VALU bound (per agent 125 instructions on weekdays,
// 381 on weekends, of which the draws 71 and 284: 32M agents in 48 replicates 102
// and 291 us; agent by agent with a check per key 10% more); the LDS adds,
// the 4-byte coalesced key stores and the row flush hide behind them.
template <bool WEEKEND>
__device__ __forceinline__ void count_block(int block, DayState* __restrict__ sts, const Model* __restrict__ models,
                                            const uint8_t* __restrict__ ages, const CountTable& T) {
    extern __shared__ uint32_t s_cnt[];
    const CountBlock blk = T.chunks[block];
    DayState* st = sts + blk.r;
    if (st->done) return;
    const Model& M = models[blk.r];
    const CountRep c = T.reps[blk.r];
    const int tid = threadIdx.x, nt = blockDim.x;
    __shared__ __align__(16) WalkRow s_row[kWalkRows];
    const LdsWalk wk = load_walk(WEEKEND ? M.we_table : M.wd_table, s_row);
    for (int i = tid; i < c.K; i += nt) s_cnt[i] = 0;
    __syncthreads();
    const int64_t N = M.N;
    const int64_t a0 = (int64_t)blk.at * c.A, a1 = min(N, a0 + c.A);  // even a0
    const uint64_t eoff = st->rand_offset;  // the day's errand offset: it moves at the day's end
    // Two agents per thread and turn; their keys, all in range unless the model
    // is at fault, are checked together.
    bool bad = false;
    auto add = [&](bool there, uint32_t k) {
        if (there) atomicAdd(&s_cnt[k], 1u);
    };
    if (WEEKEND) {
        const int base = M.we_base;
        const uint32_t E = (uint32_t)M.we_E;
        uint32_t* out = reinterpret_cast<uint32_t*>(T.keys + c.abase);
        for (int64_t g = a0 / 2 + tid; 2 * g < a1; g += nt) {
            const bool two = 2 * g + 1 < a1;
            uint32_t k[2][3];
            int32_t hour[2][3], loc[2][3];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                weekend_errands(M, wk, eoff + (uint64_t)(int64_t)(2 * ((int32_t)(2 * g) + i)), hour[i], loc[i]);
            const bool ok = weekend_pair_keys(base, E, hour, loc, two, k);
#pragma unroll
            for (int e = 0; e < 3; ++e)
                out[e * (T.slots / 2) + g] = (k[0][e] & 0xFFFFu) | (two ? k[1][e] << 16 : kNoKey << 16);
            if (ok) {
#pragma unroll
                for (int e = 0; e < 3; ++e) {
                    add(true, k[0][e]);
                    add(two, k[1][e]);
                }
            } else {
                bad = true;
            }
        }
    } else {
        const WeekdayHours hours{M.wd_base, M.wd_base1, (uint32_t)M.wd_E, (uint32_t)M.wd_E1};
        const uint8_t* age = ages + c.abase;
        uint32_t* out0 = reinterpret_cast<uint32_t*>(T.keys + c.abase);
        uint32_t* out1 = reinterpret_cast<uint32_t*>(T.keys + T.slots + c.abase);
        for (int64_t g = a0 / 2 + tid; 2 * g < a1; g += nt) {
            const bool two = 2 * g + 1 < a1;
            // (ages are padded to whole pairs)
            const uint32_t age2 = *reinterpret_cast<const uint16_t*>(age + 2 * g);
            const U4 u = draw4(eoff + (uint64_t)g, M.key0, M.key1);
            uint32_t k0[2], k1[2];
            int32_t d1[2], d2[2];
            bool adult[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                adult[i] = (i == 0 || two) && ((age2 >> (8 * i)) & 0xFFu) == kAgeAdult;
                weekday_dests(M, wk, u.w[2 * i], u.w[2 * i + 1], adult[i], d1[i], d2[i]);
            }
            const bool ok = weekday_pair_keys(hours, d1, d2, adult, two, k0, k1);
            out0[g] = (k0[0] & 0xFFFFu) | (k0[1] << 16);
            out1[g] = (k1[0] & 0xFFFFu) | (k1[1] << 16);
            if (ok) {
                add(true, k0[0]);
                add(two, k0[1]);
                add(adult[0], k1[0]);
                add(adult[1], k1[1]);
            } else {
                bad = true;
            }
        }
    }
    if (bad) st->fault = 1;
    __syncthreads();
    uint32_t* row = T.cnt + c.mbase + (int64_t)blk.at * c.K;
    for (int i = tid; i < c.K; i += nt) row[i] = s_cnt[i];
}

template <bool WEEKEND>
__global__ __launch_bounds__(1024) void k_count(const int32_t* __restrict__ done, DayState* __restrict__ sts,
                                                const Model* __restrict__ models, const uint8_t* __restrict__ ages,
                                                CountTable T) {
    if (*done) return;
    count_block<WEEKEND>(blockIdx.x, sts, models, ages, T);
}

// Column prefixes of the count matrices, kScanCols buckets per block of 1024
// threads: the row groups sum up to 8 rows each in registers, and the
// prefixes go out through LDS as runs of consecutive chunks.  The fewer
// chunks, the more buckets per block (CountPlan::scan_cols).  Also clears the
// day's marks.
constexpr int kCountScanThreads = 1024, kScanRows = 8;
template <int kScanCols>
__device__ __forceinline__ void scan_block(int block, int blocks, const DayState* __restrict__ sts,
                                           const CountTable& T) {
    for (int64_t i = (int64_t)block * blockDim.x + threadIdx.x; i < T.mark_words; i += (int64_t)blocks * blockDim.x)
        T.marks[i] = 0u;
    const CountBlock blk = T.scans ? T.scans[block] : CountBlock{0, block * kScanCols};
    if (sts[blk.r].done) return;
    const CountRep c = T.reps[blk.r];
    constexpr int kScanGroups = kCountScanThreads / kScanCols;
    constexpr int RT = kScanGroups * kScanRows;  // rows per turn
    __shared__ uint32_t s_sum[kScanGroups][kScanCols];
    __shared__ uint32_t s_pre[kScanCols][RT + 1];
    const int col = threadIdx.x % kScanCols, grp = threadIdx.x / kScanCols;
    const int b = blk.at + col;
    const uint32_t* m = T.cnt + c.mbase + b;
    uint32_t* out = T.pre + c.mbase + (int64_t)blk.at * (c.C + 1);
    const int cols = min(kScanCols, c.K - blk.at);
    uint32_t carry = 0;
    for (int s0 = 0; s0 < c.C; s0 += RT) {
        const int rows = min(c.C - s0, RT);
        const int per = (rows + kScanGroups - 1) / kScanGroups;
        const int r0 = grp * per, r1 = min(rows, r0 + per);
        uint32_t v[kScanRows], sum = 0;
#pragma unroll
        for (int i = 0; i < kScanRows; ++i) {
            v[i] = r0 + i < r1 && col < cols ? m[(int64_t)(s0 + r0 + i) * c.K] : 0u;
            sum += v[i];
        }
        s_sum[grp][col] = sum;
        __syncthreads();
        uint32_t run = carry;
#pragma unroll
        for (int g = 0; g < kScanGroups; ++g) {
            const uint32_t x = s_sum[g][col];
            if (g < grp) run += x;
            carry += x;
        }
#pragma unroll
        for (int i = 0; i < kScanRows; ++i) {
            if (r0 + i < r1) s_pre[col][r0 + i] = run;
            run += v[i];
        }
        __syncthreads();
        const bool last = s0 + RT >= c.C;
        if (last && grp == 0) s_pre[col][rows] = carry;
        __syncthreads();
        const int len = rows + (last ? 1 : 0);  // the total ends the row
        for (int i = threadIdx.x; i < cols * len; i += kCountScanThreads) {
            const int q = i / len, k = i % len;
            out[(int64_t)q * (c.C + 1) + s0 + k] = s_pre[q][k];
        }
        __syncthreads();
    }
    if (grp == 0 && col < cols) {
        T.total[c.tbase + b] = carry;
        if (carry == 1) T.lone_day[blk.r] = sts[blk.r].day + 1;
    }
}
template <int kScanCols>
__global__ __launch_bounds__(kCountScanThreads) void k_count_scan(const int32_t* __restrict__ done,
                                                                  const DayState* __restrict__ sts, CountTable T) {
    if (*done) return;
    if (blockIdx.x == 0 && threadIdx.x < 3) T.n[threadIdx.x] = 0u;  // no picks, infectors or lists yet
    scan_block<kScanCols>(blockIdx.x, gridDim.x, sts, T);
}

// Least contact count of an infector (may_infect): its household, its
// workplace unless some workplace has one person only, and its two errands
// (every errand profile has two) unless some bucket of the day has, or that is
// not known yet (counted false).
__device__ __forceinline__ int least_contacts(const CountTable& T, AgentRecord a, int r, int day, bool weekend,
                                              bool counted = true) {
    int k = record_household_size(a) > 1 ? 3 : 0;
    if (!weekend && !T.wp_lone[r]) k += record_workplace_contacts(a);
    if (counted && T.lone_day[r] != day + 1) k += 2;
    return max(k, 1);
}

// Lists the ids of the chunk's marked buckets: reserves each bucket's part of
// the chunk's share of the list, then goes through the keys, eight per load.
// The list positions are LDS counters (all ones: not marked); counters in
// global memory would need a device-scope fence here, which writes back L2
// on this GPU (41 us per day instead of 12 at 2.35M agents).
template <bool WEEKEND>
__global__ __launch_bounds__(1024) void k_collect(const int32_t* __restrict__ done,
                                                  const DayState* __restrict__ sts,
                                                  const Model* __restrict__ models, CountTable T) {
    constexpr int KPA = WEEKEND ? 3 : 2;
    load_arguments<5>();
    load_together(*done, T.chunks[blockIdx.x].r, T.chunk_day[blockIdx.x], T.reps[0].K);
    if (*done) return;
    extern __shared__ uint32_t s_cur[];
    __shared__ uint32_t s_top;
    const CountBlock blk = T.chunks[blockIdx.x];
    const DayState& st = sts[blk.r];
    const CountRep c = T.reps[blk.r];
    if (st.done || T.chunk_day[c.chunk0 + blk.at] != st.day + 1) return;
    const int tid = threadIdx.x, nt = blockDim.x;
    const uint32_t* marks = T.marks + c.qbase + (int64_t)blk.at * c.qw;
    const int64_t a0 = (int64_t)blk.at * c.A, a1 = min((int64_t)models[blk.r].N, a0 + c.A);
    uint32_t* start = T.cnt + c.mbase + (int64_t)blk.at * c.K;  // (the prefixes hold the counts now)
    if (tid == 0) s_top = (uint32_t)(KPA * (c.abase + a0));
    for (int i = tid; i < c.K; i += nt) s_cur[i] = ~0u;
    __syncthreads();
    for (int i = tid; i < c.qw; i += nt) {
        uint32_t w = marks[i];
        while (w) {
            const int b = i * 32 + __ffs(w) - 1;
            w &= w - 1;
            start[b] = s_cur[b] = atomicAdd(&s_top, start[b]);
        }
    }
    __syncthreads();
    for (int e = 0; e < KPA; ++e) {
        // (a0 is a multiple of 8 and so is the plane stride; the last words
        // may hold keys past a1)
        const uint4* keys = reinterpret_cast<const uint4*>(T.keys + e * T.slots + c.abase);
        for (int64_t g = a0 / 8 + tid; 8 * g < a1; g += nt) {
            const uint4 v = keys[g];
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint32_t key = (w[k / 2] >> (16 * (k % 2))) & 0xFFFFu;
                if (key < (uint32_t)c.K && 8 * g + k < a1 && s_cur[key] != ~0u)
                    T.list[atomicAdd(&s_cur[key], 1u)] = (int32_t)(8 * g + k);
            }
        }
    }
}

// ---- split layouts (more than kCountMaxK buckets; one simulation) ----

constexpr int kTileAgents = 4096;  // group lists: agents per tile, ids within it 12 bits
constexpr int kTileBits = 12;
static_assert(kCountMaxRanges * kCountMaxK < (1 << (32 - kTileBits)), "a pair holds any location, and none is all ones");
constexpr int kTileThreads = 512;
constexpr int kTileGroups = 96;    // at most 10 hours x kCountMaxRanges, and the end

// Weekday keys by hour, a pair of agents per thread and turn (one group per
// hour).  VALU bound: 50M agents 160 us, of which the draws 99; the walk rows
// in LDS (load_walk) took it from 184.
__global__ __launch_bounds__(256) void k_keys_weekday(DayState* __restrict__ st, const Model* __restrict__ Mp,
                                                      const uint8_t* __restrict__ age, CountTable T) {
    if (st->done) return;
    const Model& M = *Mp;
    const int64_t N = M.N;
    __shared__ __align__(16) WalkRow s_row[kWalkRows];
    const LdsWalk wk = load_walk(M.wd_table, s_row);
    __syncthreads();
    const int base = M.wd_base, base1 = M.wd_base1;
    const uint64_t eoff = st->rand_offset;
    uint32_t* const keys0 = reinterpret_cast<uint32_t*>(T.keys);
    uint32_t* const keys1 = reinterpret_cast<uint32_t*>(T.keys + T.slots);
    bool bad = false;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; 2 * g < N; g += stride) {
        const U4 u = draw4(eoff + (uint64_t)g, M.key0, M.key1);
        uint32_t w0 = 0, w1 = 0;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int64_t p = 2 * g + k;
            const bool adult = p < N && age[p] == kAgeAdult;
            int32_t d1, d2;
            weekday_dests(M, wk, u.w[2 * k], u.w[2 * k + 1], adult, d1, d2);
            bad |= ((uint32_t)(d1 - base) >= (uint32_t)M.wd_E) | (adult & ((uint32_t)(d2 - base1) >= (uint32_t)M.wd_E1));
            w0 |= ((uint32_t)(d1 - base) & 0xFFFFu) << (16 * k);
            w1 |= (adult ? (uint32_t)(d2 - base1) & 0xFFFFu : kNoKey) << (16 * k);
        }
        // (slots is a multiple of 8: the pair's store stays inside the plane)
        keys0[g] = w0;
        keys1[g] = w1;
    }
    if (bad) st->fault = 1;
}

// Pairs by group: a block draws a tile's errands and writes them grouped
// (location within the hour << kTileBits | id within the tile), staged in LDS
// so that the stores are contiguous.  VALU bound like k_count; the rank of a
// pair within its group is a returning LDS add, its order is free.  50M agents,
// weekend 545 us, of which the draws 395.
//
// Grouping by range and not by hour alone: each block of k_count_group reads
// its own pairs instead of its hour's (24M agents with 10 times the locations,
// weekend: counts 205 -> 112 us).
template <bool WEEKEND>
__global__ __launch_bounds__(kTileThreads) void k_keys_lists(DayState* __restrict__ st, const Model* __restrict__ Mp,
                                                             const uint8_t* __restrict__ age, CountTable T) {
    if (st->done) return;
    constexpr int KPA = WEEKEND ? 3 : 2, PER = kTileAgents / kTileThreads;
    __shared__ uint32_t s_stage[KPA * kTileAgents];
    __shared__ uint32_t s_cnt[kTileGroups], s_base[kTileGroups];
    const Model& M = *Mp;
    const int tid = threadIdx.x;
    const int64_t t0 = (int64_t)blockIdx.x * kTileAgents;
    __shared__ __align__(16) WalkRow s_row[kWalkRows];
    const LdsWalk wk = load_walk(WEEKEND ? M.we_table : M.wd_table, s_row);
    if (tid < kTileGroups) s_cnt[tid] = 0;
    const int ranges = T.reps[0].ranges, W = T.reps[0].W, G = T.reps[0].G;
    __syncthreads();
    const uint64_t eoff = st->rand_offset;
    uint32_t pair[KPA * PER], at[KPA * PER];
    bool bad = false;
    auto add = [&](int slot, int hour, uint32_t l, int id) {
        int g = hour * ranges;
        for (int r = 1; r < ranges; ++r) g += l >= (uint32_t)(r * W);
        pair[slot] = (l << kTileBits) | (uint32_t)id;
        at[slot] = ((uint32_t)g << 16) | atomicAdd(&s_cnt[g], 1u);
    };
#pragma unroll
    for (int i = 0; i < KPA * PER; ++i) at[i] = ~0u;
    if constexpr (WEEKEND) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int id = i * kTileThreads + tid;
            const int64_t p = t0 + id;
            int32_t hour[3], loc[3];
            if (p < M.N) {
                weekend_errands(M, wk, eoff + (uint64_t)(int64_t)(2 * (int32_t)p), hour, loc);
#pragma unroll
                for (int e = 0; e < 3; ++e) {
                    uint32_t l = (uint32_t)(loc[e] - M.we_base);
                    if (l >= (uint32_t)M.we_E) bad = true, l = 0;
                    add(3 * i + e, hour[e], l, id);
                }
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < PER / 2; ++i) {
            const int64_t g = t0 / 2 + i * kTileThreads + tid;
            if (2 * g >= M.N) continue;
            const U4 u = draw4(eoff + (uint64_t)g, M.key0, M.key1);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int64_t p = 2 * g + k;
                const int id = (int)(p - t0);
                if (p >= M.N) continue;
                const bool adult = age[p] == kAgeAdult;
                int32_t d1, d2;
                weekday_dests(M, wk, u.w[2 * k], u.w[2 * k + 1], adult, d1, d2);
                uint32_t l = (uint32_t)(d1 - M.wd_base);
                if (l >= (uint32_t)M.wd_E) bad = true, l = 0;
                add(4 * i + 2 * k, 0, l, id);
                if (adult) {
                    l = (uint32_t)(d2 - M.wd_base1);
                    if (l >= (uint32_t)M.wd_E1) bad = true, l = 0;
                    add(4 * i + 2 * k + 1, 1, l, id);
                }
            }
        }
    }
    if (bad) st->fault = 1;
    __syncthreads();
    if (tid <= G) {
        uint32_t b = 0;
        for (int h = 0; h < tid; ++h) b += s_cnt[h];
        s_base[tid] = b;
        T.tile_off[(int64_t)blockIdx.x * T.reps[0].toff + tid] = (uint16_t)b;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KPA * PER; ++i)
        if (at[i] != ~0u) s_stage[s_base[at[i] >> 16] + (at[i] & 0xFFFFu)] = pair[i];
    __syncthreads();
    const int n = (int)s_base[G];
    uint32_t* out = T.keys32 + KPA * t0;
    for (int i = tid; i < n; i += kTileThreads) out[i] = s_stage[i];
}

// Calls f(location within the hour, agent) for the pairs of the chunk's groups
// [g0, g1) in part `part` of `parts`.  L: keys per agent of the group lists,
// or 0: 2-byte keys by hour.
template <int L, class F>
__device__ __forceinline__ void group_pairs(const CountTable& T, const CountRep& c, int64_t N, int chunk, int g0, int g1,
                                            int part, int parts, F f) {
    const int64_t a0 = (int64_t)chunk * c.A, a1 = min(N, a0 + c.A);
    const int tid = threadIdx.x, nt = blockDim.x;
    if constexpr (L > 0) {
        // A wave per tile.
        const int lane = tid & 63, waves = nt >> 6;
        const int t1 = (int)((a1 + kTileAgents - 1) / kTileAgents);
        for (int t = (int)(a0 / kTileAgents) + part * waves + (tid >> 6); t < t1; t += parts * waves) {
            const uint16_t* o = T.tile_off + (int64_t)t * c.toff;
            const int b = o[g0], e = o[g1];
            const uint32_t* src = T.keys32 + (int64_t)t * L * kTileAgents;
            constexpr int U = 8;
            for (int i0 = b; i0 < e; i0 += U * 64) {
                uint32_t v[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int i = i0 + u * 64 + lane;
                    v[u] = i < e ? src[i] : ~0u;
                }
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (v[u] != ~0u)
                        f(v[u] >> kTileBits, t * kTileAgents + (int)(v[u] & ((1u << kTileBits) - 1u)));
            }
        }
    } else {
        const uint16_t* keys = T.keys + g0 * T.slots;
        constexpr int U = 4;
        for (int64_t w0 = a0 / 8 + (int64_t)part * U * nt + tid; w0 * 8 < a1; w0 += (int64_t)parts * U * nt) {
            uint4 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t w = w0 + (int64_t)u * nt;
                v[u] = w * 8 < a1 ? reinterpret_cast<const uint4*>(keys)[w] : make_uint4(~0u, ~0u, ~0u, ~0u);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t p0 = (w0 + (int64_t)u * nt) * 8;
                const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const uint32_t key = (w[k / 2] >> (16 * (k % 2))) & 0xFFFFu;
                    if (key != kNoKey && p0 + k < a1) f(key, (int)(p0 + k));
                }
            }
        }
    }
}

// Group g of chunk: its hour, first location there, locations, and first
// bucket.  (A narrow hour leaves its last groups empty: the groups of all hours
// are as wide as the widest's need.)
struct GroupColumns {
    int hour, lo, n, bucket;
};
// An hour ends where the next begins, the last at K.
__host__ __device__ inline int hour_end(const CountRep& c, int hour) {
    return hour == c.G / c.ranges - 1 ? c.K : (hour + 1) * c.E;
}
__host__ __device__ inline GroupColumns group_columns(const CountRep& c, int g) {
    GroupColumns q;
    q.hour = g / c.ranges;
    q.lo = (g % c.ranges) * c.W;
    q.bucket = q.hour * c.E + q.lo;
    const int left = hour_end(c, q.hour) - q.bucket;
    q.n = left < 0 ? 0 : (left < c.W ? left : c.W);
    return q;
}

// All groups of an hour.
__host__ __device__ inline GroupColumns hour_columns(const CountRep& c, int hour) {
    return GroupColumns{hour, 0, hour_end(c, hour) - hour * c.E, hour * c.E};
}

// The mark words that hold q's buckets: [first, end), none if it has none.
__host__ __device__ inline int first_mark_word(const GroupColumns& q) { return q.bucket / 32; }
__host__ __device__ inline int end_mark_word(const GroupColumns& q) {
    return q.n > 0 ? (q.bucket + q.n + 31) / 32 : first_mark_word(q);
}

// Counts of a (chunk, group).  Bound by reading its keys (16 bytes per lane
// and load) or pairs; LDS adds hide behind them: 50M agents, 40 us per weekday
// (5 TB/s), 163 us per weekend day (3.7 TB/s).
template <int L>
__global__ __launch_bounds__(1024) void k_count_group(const DayState* __restrict__ st, const Model* __restrict__ Mp,
                                                      CountTable T) {
    if (st->done) return;
    extern __shared__ uint32_t s_cnt[];
    const CountRep c = T.reps[0];
    const int chunk = blockIdx.x / c.G, g = blockIdx.x % c.G;
    const GroupColumns q = group_columns(c, g);
    const int tid = threadIdx.x, nt = blockDim.x;
    for (int i = tid; i < q.n; i += nt) s_cnt[i] = 0;
    __syncthreads();
    group_pairs<L>(T, c, Mp->N, chunk, g, g + 1, 0, 1, [&](uint32_t l, int) {
        const uint32_t i = l - (uint32_t)q.lo;
        if (i < (uint32_t)q.n) atomicAdd(&s_cnt[i], 1u);
    });
    __syncthreads();
    uint32_t* row = T.cnt + c.mbase + (int64_t)chunk * c.K + q.bucket;
    for (int i = tid; i < q.n; i += nt) row[i] = s_cnt[i];
}

// Lists of a (chunk, group)'s marked buckets, reserved with their first marks
// (the count matrix holds each list's start, and its end once collected).
// Up to kFewMarks marks per group of an hour, kCollectParts small blocks share
// the hour's keys and append with atomics on the matrix; above, a block per
// group appends with LDS counters.  Both are bound by reading the hour's keys:
// 50M agents, a weekday with few marks 29 us (7 TB/s, one block per group 109
// us), with many 65 us; 8 parts of 256 threads: the same on weekdays, 155 us
// instead of 98-140 on weekends of up to 96 marks.
constexpr uint32_t kFewMarks = 96;
constexpr int kCollectParts = 16, kCollectFewThreads = 512;

// Marked buckets of the group, by the whole block; f(bucket) for each.
template <class F>
__device__ __forceinline__ void for_marked(const uint32_t* __restrict__ marks, const GroupColumns& q, F f) {
    for (int i = first_mark_word(q) + threadIdx.x; i < end_mark_word(q); i += blockDim.x) {
        uint32_t w = marks[i];
        while (w) {
            const int b = i * 32 + __ffs(w) - 1;
            w &= w - 1;
            if (b >= q.bucket && b < q.bucket + q.n) f(b);
        }
    }
}

template <int L>
__global__ __launch_bounds__(kCollectFewThreads) void k_collect_few(const DayState* __restrict__ st,
                                                                    const Model* __restrict__ Mp, CountTable T) {
    if (st->done) return;
    const CountRep c = T.reps[0];
    // (chunk, hour): the hour's groups share one pass over its keys
    const int ch = blockIdx.x / kCollectParts, part = blockIdx.x % kCollectParts;
    bool any = false;
    for (int g = 0; g < c.ranges; ++g) any |= T.chunk_day[ch * c.ranges + g] == st->day + 1;
    if (!any) return;
    extern __shared__ uint32_t s_bits[];
    __shared__ uint32_t s_n;
    const int hours = c.G / c.ranges, chunk = ch / hours, tid = threadIdx.x;
    const GroupColumns q = hour_columns(c, ch % hours);
    for (int i = tid; i < (q.n + 31) / 32; i += blockDim.x) s_bits[i] = 0;
    if (tid == 0) s_n = 0;
    __syncthreads();
    for_marked(T.marks + c.qbase + (int64_t)chunk * c.qw, q, [&](int b) {
        atomicAdd(&s_n, 1u);
        atomicOr(&s_bits[(b - q.bucket) >> 5], 1u << ((b - q.bucket) & 31));
    });
    __syncthreads();
    if (s_n > kFewMarks * (uint32_t)c.ranges) return;
    uint32_t* cursor = T.cnt + c.mbase + (int64_t)chunk * c.K + q.bucket;
    group_pairs<L>(T, c, Mp->N, chunk, q.hour * c.ranges, (q.hour + 1) * c.ranges, part, kCollectParts,
                   [&](uint32_t l, int p) {
                       const uint32_t i = l - (uint32_t)q.lo;
                       if (i < (uint32_t)q.n && is_marked(s_bits, i)) T.list[atomicAdd(&cursor[i], 1u)] = p;
                   });
}

template <int L>
__global__ __launch_bounds__(1024) void k_collect_group(const DayState* __restrict__ st, const Model* __restrict__ Mp,
                                                        CountTable T) {
    if (st->done) return;
    const CountRep c = T.reps[0];
    if (T.chunk_day[blockIdx.x] != st->day + 1) return;
    extern __shared__ uint32_t s_cur[];
    __shared__ uint32_t s_n;
    const int chunk = blockIdx.x / c.G, g = blockIdx.x % c.G;
    const GroupColumns q = group_columns(c, g);
    const int tid = threadIdx.x, nt = blockDim.x;
    const uint32_t* marks = T.marks + c.qbase + (int64_t)chunk * c.qw;
    uint32_t* cursor = T.cnt + c.mbase + (int64_t)chunk * c.K + q.bucket;
    if (tid == 0) s_n = 0;
    __syncthreads();
    for_marked(marks, hour_columns(c, q.hour), [&](int) { atomicAdd(&s_n, 1u); });
    __syncthreads();
    if (s_n <= kFewMarks * (uint32_t)c.ranges) return;
    for (int i = tid; i < q.n; i += nt) s_cur[i] = ~0u;
    __syncthreads();
    for_marked(marks, q, [&](int b) { s_cur[b - q.bucket] = cursor[b - q.bucket]; });
    __syncthreads();
    group_pairs<L>(T, c, Mp->N, chunk, g, g + 1, 0, 1, [&](uint32_t l, int p) {
        const uint32_t i = l - (uint32_t)q.lo;
        if (i < (uint32_t)q.n && s_cur[i] != ~0u) T.list[atomicAdd(&s_cur[i], 1u)] = p;
    });
    __syncthreads();
    for_marked(marks, q, [&](int b) { cursor[b - q.bucket] = s_cur[b - q.bucket]; });
}

// Short lists rank every id against the others, in registers;
// longer ones (few buckets, at least 1,024 agents per chunk) bisect the
// chunk's id range (at most 15 steps of len / 16 loads).
constexpr int kPickLanes = 16;
constexpr uint32_t kRankByCount = 64;

// 16 lanes: the id with `want` smaller ones among the len distinct ids of l,
// all in [a0, a0 + A).
__device__ __forceinline__ int32_t rank_in_list(const int32_t* __restrict__ l, uint32_t len, uint32_t want, int32_t a0,
                                                int32_t A, int sub) {
    if (len <= kRankByCount) {
        constexpr int R = kRankByCount / kPickLanes;
        int32_t x[R];
        uint32_t rank[R];
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const uint32_t t = sub + i * kPickLanes;
            x[i] = t < len ? l[t] : 0x7FFFFFFF;
            rank[i] = 0;
        }
#pragma unroll
        for (int i = 0; i < R; ++i) {
            if (i * kPickLanes >= (int)len) break;
#pragma unroll
            for (int t = 0; t < kPickLanes; ++t) {
                const int32_t y = __shfl(x[i], t, kPickLanes);
#pragma unroll
                for (int k = 0; k < R; ++k) rank[k] += y < x[k];
            }
        }
        int32_t found = -1;
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (rank[i] == want && x[i] != 0x7FFFFFFF) found = x[i];
#pragma unroll
        for (int o = kPickLanes / 2; o > 0; o >>= 1) found = max(found, __shfl_xor(found, o, kPickLanes));
        return found;
    }
    // The smallest id with more than `want` ids at or below it.
    int32_t lo = a0, hi = a0 + A - 1;
    while (lo < hi) {
        const int32_t mid = lo + ((hi - lo) >> 1);
        uint32_t le = 0;
        for (uint32_t i = sub; i < len; i += kPickLanes) le += l[i] <= mid;
#pragma unroll
        for (int o = kPickLanes / 2; o > 0; o >>= 1) le += __shfl_xor(le, o, kPickLanes);
        if (le > want)
            hi = mid;
        else
            lo = mid + 1;
    }
    return lo;
}

// 16 lanes: the agent with `want` agents of bucket b before it in the chunk,
// from the chunk's keys, 1,024 agents at a time, 64 consecutive ones per lane.
constexpr int kDirectChunk = 4096;
__device__ __forceinline__ int32_t rank_in_keys(const CountTable& T, const CountRep& c, int chunk, uint32_t b,
                                                uint32_t want, int sub) {
    constexpr int kLaneAgents = 64;
    for (int p0 = chunk * c.A + sub * kLaneAgents;; p0 += kPickLanes * kLaneAgents) {
        uint64_t m = 0;
        // (a weekday bucket's hour is its plane; weekend hours come in any order)
        const int e0 = T.direct == 2 && b >= T.hour1 ? 1 : 0, e1 = T.direct == 2 ? e0 + 1 : T.direct;
        for (int e = e0; e < e1; ++e) {
            const uint4* keys = reinterpret_cast<const uint4*>(T.keys + e * T.slots + c.abase + p0);
            uint4 v[kLaneAgents / 8];
#pragma unroll
            for (int i = 0; i < kLaneAgents / 8; ++i)
                v[i] = p0 + 8 * i < T.n_agents ? keys[i] : make_uint4(~0u, ~0u, ~0u, ~0u);
#pragma unroll
            for (int i = 0; i < kLaneAgents / 8; ++i) {
                const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
                uint32_t bits = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    bits |= ((w[k] & 0xFFFFu) == b ? 1u : 0u) << (2 * k);
                    bits |= ((w[k] >> 16) == b ? 2u : 0u) << (2 * k);
                }
                m |= (uint64_t)bits << (8 * i);
            }
        }
        const int left = T.n_agents - p0;  // keys past the last agent are left from other days
        if (left < kLaneAgents) m &= left <= 0 ? 0ull : (1ull << left) - 1ull;
        const uint32_t n = (uint32_t)__popcll(m);
        uint32_t inc = n;  // a row of 16 lanes
        inc = dpp_add<0x111>(inc);
        inc = dpp_add<0x112>(inc);
        inc = dpp_add<0x114>(inc);
        inc = dpp_add<0x118>(inc);
        int32_t found = -1;
        if (inc > want && inc - n <= want) {
            for (uint32_t t = want - (inc - n); t; --t) m &= m - 1;
            found = p0 + __ffsll((unsigned long long)m) - 1;
        }
#pragma unroll
        for (int o = kPickLanes / 2; o > 0; o >>= 1) found = max(found, __shfl_xor(found, o, kPickLanes));
        const uint32_t all = __shfl(inc, kPickLanes - 1, kPickLanes);
        if (found >= 0 || p0 - sub * kLaneAgents + kPickLanes * kLaneAgents >= (chunk + 1) * c.A) return found;
        want -= all;
    }
}

// The picked person of every queued pick and its claims (process_contacts).
constexpr uint32_t kPicksPerClaim = 64;

// 16 lanes: the person of pick q.
__device__ __forceinline__ int32_t picked_person(const CountTable& T, uint32_t q, int sub) {
    const uint32_t b = T.pk_bucket[q];
    const int32_t idx = T.pk_idx[q];
    const CountRep c = T.reps[T.pk_r[q]];
    uint32_t want = T.pk_want[q], len = (uint32_t)T.pk_len[q];
    int chunk = T.pk_chunk[q];
    for (int round = 0;; ++round) {
        int32_t v;
        if (T.direct) {
            v = rank_in_keys(T, c, chunk, b, want, sub);
        } else {
            // (split layouts: the entry is the list's end now)
            const int32_t* l = T.list + (T.cnt[c.mbase + (int64_t)chunk * c.K + b] - (c.G > 1 ? len : 0u));
            v = rank_in_list(l, len, want, chunk * c.A, c.A, sub);
        }
        if (v != idx || round) return v;
        const uint32_t total = T.total[c.tbase + b];  // the next person instead (select_person)
        uint32_t j = count_column(T, c, b)[chunk] + want + 1, before;
        if (j == total) j = 0;
        chunk = chunk_of(T, c, b, j, total, before, len);
        want = j - before;
    }
}

__global__ __launch_bounds__(256) void k_resolve(DayState* __restrict__ g, CountTable T, ClaimArrays C) {
    load_arguments<5>();
    load_together(g->done, T.n[0], T.reps[0].K, g->day);
    if (g->done) return;
    const uint32_t n = *T.n;
    const int sub = threadIdx.x % kPickLanes, lane = threadIdx.x & 63;
    // A block finds the people of `per` picks, 16 at a time, and its first
    // wave claims them together: one list atomic per `per` picks.
    const uint32_t per = n > kPicksPerClaim * gridDim.x ? kPicksPerClaim : 256 / kPickLanes;
    __shared__ int32_t s_v[kPicksPerClaim];
    for (uint32_t q0 = blockIdx.x * per; q0 < n; q0 += gridDim.x * per) {
        const uint32_t q1 = min(n, q0 + per);
        for (uint32_t q = q0 + threadIdx.x / kPickLanes; q < q1; q += 256 / kPickLanes) {
            const int32_t v = picked_person(T, q, sub);
            if (sub == 0) s_v[q - q0] = v;
        }
        __syncthreads();
        if (threadIdx.x < 64) {
            const uint32_t q = q0 + lane;
            bool newp = false, news = false;
            int64_t slot = 0;
            if (q < q1) {
                slot = T.reps[T.pk_r[q]].abase + s_v[lane];
                post_claims(C, slot, T.pk_claim[q], T.pk_payload[q], newp, news);
            }
            const uint64_t mp = __ballot(newp), ms = __ballot(news);
            uint32_t base = 0;
            if (lane < 2) {
                const uint32_t k = (uint32_t)__popcll(lane ? ms : mp);
                if (k) base = atomicAdd(&C.n_claimed[lane], k);
            }
            const uint64_t below = (1ull << lane) - 1;
            const uint32_t bp = __shfl(base, 0, 64), bs = __shfl(base, 1, 64);
            if (newp) C.list_p[bp + (uint32_t)__popcll(mp & below)] = (int32_t)slot;
            if (news) C.list_s[bs + (uint32_t)__popcll(ms & below)] = (int32_t)slot;
        }
        __syncthreads();
    }
}

}  // namespace

// ---------------- host side ----------------

// Agents per chunk for N agents, K buckets and kpa keys per agent.  About 8
// people per bucket and chunk keep the matrix at an eighth of the pairs and a
// pick's list at 8 ids; smaller chunks (down to one person per bucket)
// while there are fewer than `want` of them, to fill the chip.
inline int32_t count_chunk(int64_t N, int64_t K, int kpa, int64_t want) {
    const int64_t a = std::max<int64_t>({(int64_t)kCountMinChunk, K / kpa, std::min(8 * K / kpa, (N + want - 1) / want)});
    return (int32_t)((a + 511) / 512 * 512);
}

// The plan of one layout on the host, and its device copies.
struct CountPlan {
    bool on = false;
    bool split = false, lists = false;  // column groups; pairs in group lists
    int n_chunks = 0, n_scans = 0, threads = 0, kpa = 0, scan_cols = 0;
    size_t lds = 0;
    int64_t entries = 0, mark_words = 0, buckets = 0;
    std::vector<CountRep> reps;
    std::vector<CountBlock> chunks, scans;
    CountRep* d_reps = nullptr;
    CountBlock *d_chunks = nullptr, *d_scans = nullptr;

    // reps' K and abase are set; N per simulation.  Leaves `on` false when
    // a simulation has too many buckets for LDS, or so few for its agents
    // (over kCountMaxLen people per bucket in the smallest chunk) that lists
    // would approach the whole table.
    // At least about `want` chunks in all, if lists stay above one id.
    void build(const std::vector<int64_t>& N, int keys_per_agent, int64_t want) {
        kpa = keys_per_agent;
        int32_t kmax = 0;
        int64_t total = 0;
        for (int64_t n : N) total += n;
        on = true;
        for (size_t r = 0; r < reps.size(); ++r) {
            kmax = std::max(kmax, reps[r].K);
            if ((int64_t)kCountMinChunk * kpa > (int64_t)kCountMaxLen * reps[r].K && N[r] > kCountSmall) on = false;
        }
        on = on && kmax <= kCountMaxK;
        if (!on) return;
        for (auto& c : reps) c.G = c.ranges = 1, c.E = c.W = c.K;
        lds = sizeof(uint32_t) * (size_t)kmax;
        threads = 1024;
        for (size_t r = 0; r < reps.size(); ++r) {
            CountRep& c = reps[r];
            c.A = count_chunk(N[r], c.K, kpa, std::max<int64_t>(1, want * N[r] / total));
            c.C = (int32_t)((N[r] + c.A - 1) / c.A);
            c.qw = (c.K + 31) / 32;
            c.mbase = entries;
            c.tbase = buckets;
            buckets += c.K;
            c.qbase = mark_words;
            c.chunk0 = n_chunks;
            n_chunks += c.C;
            entries += (int64_t)(c.C + 1) * c.K;
            mark_words += (int64_t)c.C * c.qw;
        }
        // The largest first: a large block started last would run alone (48
        // replicates of 50k to 2M agents: 118 -> 102 us per weekday, 386 -> 291
        // per weekend day).
        std::vector<int32_t> order(reps.size());
        for (size_t r = 0; r < reps.size(); ++r) order[r] = (int32_t)r;
        std::stable_sort(order.begin(), order.end(), [this](int32_t x, int32_t y) { return reps[x].A > reps[y].A; });
        chunks.reserve(n_chunks);
        for (int32_t r : order)
            for (int k = 0; k < reps[r].C; ++k) chunks.push_back({r, k});
        // More chunks than CUs: the smallest blocks that still fill a CU's 2,048
        // threads beside the counters, so that one's start (counters cleared,
        // marks read) and end overlap the others' work.  48 replicates of 0.7M
        // agents, weekday lists: 62 us with 1,024 threads, 41 with 256.
        if (n_chunks > want) {
            const int64_t resident = std::max<int64_t>(1, (160 * 1024) / ((int64_t)lds + 2048));
            int64_t best = 0;
            for (int t = 1024; t >= 256; t /= 2) {
                const int64_t all = t * std::min<int64_t>(resident, 2048 / t);
                if (all >= best) best = all, threads = t;
            }
        }
        plan_scans();
    }
    // Buckets per block of k_count_scan: the fewer, the more rows (chunks) a turn
    // covers and the shorter the runs of the matrix that it reads.  64 unless a
    // block would have few rows to do (32 chunks or less: 256, 8 or less: 1,024)
    // or there would be few blocks with many (up to 128 blocks and over 128
    // chunks: 32).  us with 32 / 64 / 256 / 1,024 buckets (* taken), and where:
    //   657 chunks    870 buckets  *11 /  18 /   60 / 220  2.4M agents, location scale 0.3, weekday
    //   253         6,381           *7 /   9 /   25 /  95  5.2M, 2.2, weekday
    //   256        14,501           13 / *11 /   26 /  95  12M, 5, weekday
    //   253        28,600           24 / *16 /   27 /  95  5.2M, 2.2, weekend
    //   128        61,596           33 / *18 /   21 /  51  50M, 21.24, weekday
    //    58       116,001           46 / *19 /   15 /  27  235k, 40, weekday
    //    51       276,110          103 / *39 /   32 /  60  50M, 21.24, weekend
    //    32       290,001           98 /  32 /  *19 /  36  24M, 100, weekday
    //     6     1,300,000          387 /  99 /   32 / *19  24M, 100, weekend
    void plan_scans() {
        int32_t chunks_max = 0;
        for (const auto& c : reps) chunks_max = std::max(chunks_max, c.C);
        scan_cols = chunks_max > 128 && buckets <= 128 * 64 ? 32 : (chunks_max > 32 ? 64 : (chunks_max > 8 ? 256 : 1024));
        // One simulation's blocks need no list: at 50M agents it would be most of
        // what set-up sends (70 KB, 0.4 ms through pageable memory).
        if (reps.size() == 1) {
            n_scans = (reps[0].K + scan_cols - 1) / scan_cols;
            return;
        }
        for (size_t r = 0; r < reps.size(); ++r)
            for (int b = 0; b < reps[r].K; b += scan_cols) scans.push_back({(int32_t)r, b});
        n_scans = (int)scans.size();
    }
    // One simulation of more buckets: column groups, E locations in the first
    // hour, `hours` hours.  Chunks so that the (chunk, group) blocks fill the
    // chip once or a few times (a block may take a CU's whole LDS) with at
    // most about 16 people per bucket and chunk.
    void build_split(int64_t N, int keys_per_agent, int32_t E, int hours, int cus) {
        CountRep& c = reps[0];
        kpa = keys_per_agent;
        c.E = E;
        const int32_t last = c.K - (hours - 1) * E, widest = std::max(E, last);
        c.ranges = (widest + kCountMaxK - 1) / kCountMaxK;
        if (c.ranges > kCountMaxRanges) return;
        c.W = (widest + c.ranges - 1) / c.ranges;
        c.G = hours * c.ranges;
        int64_t A = 0;
        for (int k = 1;; ++k) {
            const int64_t C = std::max<int64_t>(1, (int64_t)cus * k / c.G);
            A = ((N + C - 1) / C + kTileAgents - 1) / kTileAgents * kTileAgents;
            if (kpa * A <= 16 * (int64_t)c.K || A == kTileAgents) break;
        }
        on = split = true;
        // Weekend hours are not in the order of the slots; a weekday hour in
        // several groups would be read by each (24M agents, 4-byte keys:
        // 84 us for them and 111 for the counts, instead of 114 and 53).
        lists = kpa == 3 || c.ranges > 1;
        c.toff = (c.G + 16) / 16 * 16;
        c.A = (int32_t)A;
        c.C = (int32_t)((N + A - 1) / A);
        c.qw = (c.K + 31) / 32;
        entries = (int64_t)(c.C + 1) * c.K;
        buckets = c.K;
        mark_words = (int64_t)c.C * c.qw;
        lds = sizeof(uint32_t) * (size_t)c.W;
        threads = 1024;
        n_chunks = c.C * c.G;
        plan_scans();
    }
    // (the device copies belong to CountScratch's block)
    void release() { *this = CountPlan(); }
};

// Buffers shared by the two layouts (weekday, weekend) and the device copies of
// their plans, in one allocation: the plans, then cleared counters, all sent in
// one copy, then the rest.  The two matrices go to one of the caller's buffers
// that is idle on counted days, if they fit: the sorted tables' digit counts, or
// `spare`.
struct CountScratch {
    unsigned char* block = nullptr;
    std::vector<unsigned char> image;  // what is sent, kept until it has been
    uint32_t *cnt = nullptr, *pre = nullptr, *total = nullptr, *marks = nullptr, *n = nullptr;
    int32_t* chunk_day = nullptr;
    uint16_t* tile_off = nullptr;
    int32_t* lone_day = nullptr;
    int alloc(CountPlan (&plan)[2], int64_t N, hipStream_t st, const TableScratch& ts, void* spare, int64_t spare_bytes) {
        const CountPlan &a = plan[0], &b = plan[1];
        const int64_t e = std::max(a.entries, b.entries);
        if (e == 0) return 0;
        size_t bytes = 0;
        const auto take = [&](size_t count, size_t size) {
            const size_t at = bytes;
            bytes += (std::max<size_t>(count, 1) * size + 255) / 256 * 256;
            return at;
        };
        size_t at_plan[2][3] = {};
        for (int w = 0; w < 2; ++w) {
            CountPlan& p = plan[w];
            if (!p.on) continue;
            at_plan[w][0] = take(p.reps.size(), sizeof(CountRep));
            at_plan[w][1] = take(p.chunks.size(), sizeof(CountBlock));
            at_plan[w][2] = take(p.scans.size(), sizeof(CountBlock));
        }
        const size_t at_n = take(4, sizeof(uint32_t)), sent = bytes;
        const size_t at_lone = take(std::max(a.reps.size(), b.reps.size()), sizeof(int32_t));
        const size_t at_day = take(std::max(a.n_chunks, b.n_chunks), sizeof(int32_t));
        const size_t at_total = take(std::max(a.buckets, b.buckets), sizeof(uint32_t));
        const size_t at_marks = take(std::max(a.mark_words, b.mark_words), sizeof(uint32_t));
        const size_t at_tile = take(a.lists || b.lists ? (N / kTileAgents + 1) *
                                        std::max(a.lists ? a.reps[0].toff : 0, b.lists ? b.reps[0].toff : 0) : 0,
                                    sizeof(uint16_t));
        const int64_t matrix = (e + 63) / 64 * 64;
        const int64_t both = 2 * matrix * (int64_t)sizeof(uint32_t);
        void* const idle = both <= ts.hist_bytes ? ts.hist : (both <= spare_bytes ? spare : nullptr);
        const size_t at_matrices = take(idle ? 0 : 2 * matrix, sizeof(uint32_t));
        if (dev_alloc(&block, (int64_t)bytes)) return PT_ENOMEM;
        image.assign(sent, 0);
        for (int w = 0; w < 2; ++w) {
            CountPlan& p = plan[w];
            if (!p.on) continue;
            memcpy(image.data() + at_plan[w][0], p.reps.data(), sizeof(CountRep) * p.reps.size());
            memcpy(image.data() + at_plan[w][1], p.chunks.data(), sizeof(CountBlock) * p.chunks.size());
            memcpy(image.data() + at_plan[w][2], p.scans.data(), sizeof(CountBlock) * p.scans.size());
            p.d_reps = (CountRep*)(block + at_plan[w][0]);
            p.d_chunks = (CountBlock*)(block + at_plan[w][1]);
            p.d_scans = p.scans.empty() ? nullptr : (CountBlock*)(block + at_plan[w][2]);
        }
        HIP_TRY(hipMemcpyAsync(block, image.data(), sent, hipMemcpyHostToDevice, st));
        n = (uint32_t*)(block + at_n);
        lone_day = (int32_t*)(block + at_lone);
        chunk_day = (int32_t*)(block + at_day);
        total = (uint32_t*)(block + at_total);
        marks = (uint32_t*)(block + at_marks);
        tile_off = (uint16_t*)(block + at_tile);
        cnt = idle ? (uint32_t*)idle : (uint32_t*)(block + at_matrices);
        pre = cnt + matrix;
        return 0;
    }
    void release() {
        dev_free(block);
        *this = CountScratch();
    }
    void fill(CountTable& t, const CountPlan& p) const {
        t.reps = p.d_reps;
        t.chunks = p.d_chunks;
        t.scans = p.d_scans;
        t.cnt = cnt;
        t.pre = pre;
        t.total = total;
        t.marks = marks;
        t.mark_words = p.mark_words;
        t.chunk_day = chunk_day;
        t.n = n;
        t.tile_off = tile_off;
        t.lone_day = lone_day;
    }
};

// LDS above the default limit for the counting kernels.
inline hipError_t set_count_lds(const CountPlan& p) {
    if (!p.on || p.lds <= 64 * 1024) return hipSuccess;
    const auto ptr = [](auto* k) { return reinterpret_cast<const void*>(k); };
    for (const void* k :
         {ptr(&k_count<false>), ptr(&k_count<true>), ptr(&k_collect<false>), ptr(&k_collect<true>),
          ptr(&k_count_group<0>), ptr(&k_count_group<2>), ptr(&k_count_group<3>), ptr(&k_collect_group<0>),
          ptr(&k_collect_group<2>), ptr(&k_collect_group<3>)}) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(4 * kCountMaxK));
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Before contacts: keys, counts, prefixes.  After: lists, picks, claims.
inline void enqueue_counts(const CountPlan& p, const CountTable& t, const int32_t* done, DayState* sts,
                           const Model* models, const uint8_t* age, bool weekend, hipStream_t st, LaunchTimer* tm,
                           int64_t models_n = 0, int grid_keys = 0) {
    if (p.split) {
        const int64_t N = models_n;
        if (p.lists)
            launch(tm, weekend ? KC_GEN_WEEKEND : KC_GEN_WEEKDAY, weekend ? k_keys_lists<true> : k_keys_lists<false>,
                   dim3((int)((N + kTileAgents - 1) / kTileAgents)), dim3(kTileThreads), st, sts, models, age, t);
        else
            launch(tm, KC_GEN_WEEKDAY, k_keys_weekday, dim3(grid_for((N + 1) / 2, 256, grid_keys)), dim3(256), st, sts,
                   models, age, t);
        const auto k = weekend ? k_count_group<3> : (p.lists ? k_count_group<2> : k_count_group<0>);
        launch_lds(tm, KC_TABLE_COUNT, k, dim3(p.n_chunks), dim3(p.threads), p.lds, st, (const DayState*)sts, models, t);
    } else {
        launch_lds(tm, weekend ? KC_GEN_WEEKEND : KC_GEN_WEEKDAY, weekend ? k_count<true> : k_count<false>,
                   dim3(p.n_chunks), dim3(p.threads), p.lds, st, done, sts, models, age, t);
    }
    const auto scan = p.scan_cols == 32
                          ? k_count_scan<32>
                          : (p.scan_cols == 64 ? k_count_scan<64> : (p.scan_cols == 256 ? k_count_scan<256> : k_count_scan<1024>));
    launch(tm, KC_COUNT_SCAN, scan, dim3(p.n_scans), dim3(kCountScanThreads), st, done, (const DayState*)sts, t);
}

inline void enqueue_picks(const CountPlan& p, const CountTable& t, const ClaimArrays& c, DayState* g,
                          const DayState* sts, const Model* models, int grid, bool weekend, hipStream_t st,
                          LaunchTimer* tm) {
    if (p.split) {
        const auto few = weekend ? k_collect_few<3> : (p.lists ? k_collect_few<2> : k_collect_few<0>);
        launch_lds(tm, KC_COLLECT, few, dim3(p.n_chunks / p.reps[0].ranges * kCollectParts), dim3(kCollectFewThreads),
                   sizeof(uint32_t) * (size_t)(p.reps[0].W * p.reps[0].ranges / 32 + 2), st, sts, models, t);
        const auto k = weekend ? k_collect_group<3> : (p.lists ? k_collect_group<2> : k_collect_group<0>);
        launch_lds(tm, KC_COLLECT, k, dim3(p.n_chunks), dim3(p.threads), p.lds, st, sts, models, t);
    } else if (!t.direct) {
        launch_lds(tm, KC_COLLECT, weekend ? k_collect<true> : k_collect<false>, dim3(p.n_chunks), dim3(p.threads),
                   p.lds, st, (const int32_t*)&g->done, sts, models, t);
    }
    launch(tm, KC_RESOLVE, k_resolve, dim3(grid), dim3(256), st, g, t, c);
}

}  // namespace pt
