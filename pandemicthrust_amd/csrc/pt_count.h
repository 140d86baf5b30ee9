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
//   k_count_scan  per bucket, the exclusive prefix over the chunks (in
//                 place) and the total: pre[c][b] people of bucket b lie in
//                 chunks before c
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
// A chunk's list order does not matter (ranks are taken by value), so the
// result is the id the sorted table holds at that position.
//
// Used for layouts of at most kCountMaxK buckets (32-bit counters in one
// CU's 160 KB LDS).
//
// Citations are relative to PandemicThrust/PandemicThrust/ of the reference.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "pt_day.h"

namespace pt {

constexpr int kCountMaxK = 40000;       // 32-bit counters: 160,000 of the 163,840 bytes of LDS
constexpr uint32_t kNoKey = 0xFFFFu;    // no pair (weekday hour 1 of a child)
constexpr int kCountMinChunk = 1024;    // agents
constexpr int kCountMaxLen = 64;        // people per bucket of a smallest chunk (CountPlan::build)
constexpr int64_t kCountSmall = 1000000;  // agents up to which the lists' length does not matter

// One simulation's counted table in one layout (weekday or weekend).
struct CountRep {
    int64_t abase;  // first agent slot
    int64_t mbase;  // first entry of its (C + 1) x K matrix (row C: totals)
    int64_t qbase;  // first word of its C x qw mark words
    int32_t K, C, A, qw;  // buckets, chunks, agents per chunk, mark words per chunk
    int32_t chunk0; // first chunk (k_count block)
    int32_t pad;
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
    const CountBlock* scans;
    uint16_t* keys;        // keys per agent x slots
    int64_t slots;
    uint32_t* pre;         // the matrices
    uint32_t* cursor;      // same shape: list positions of marked (chunk, bucket)
    uint32_t* marks;       // mark words
    int64_t mark_words;
    int32_t* chunk_day;    // day + 1 on which the chunk was last marked
    int32_t* list;         // ids of the marked buckets, kpa * agents per chunk
    uint32_t* n;           // [0] picks queued, [1] infectors listed
    // Listed infectors: agent, position, pack_infectivity, simulation (batch).
    int32_t *sv_idx, *sv_pos;
    uint32_t* sv_f;
    int32_t* sv_r;
    uint32_t *pk_bucket, *pk_want, *pk_claim, *pk_payload;  // queued picks: rank `want` of
    int32_t *pk_idx, *pk_r, *pk_chunk, *pk_len;             // the len ids of (chunk, bucket)
};

__host__ __device__ inline ClaimArrays claim_arrays(const AgentArrays& A, int32_t* list_p, int32_t* list_s,
                                                    uint32_t* n_claimed) {
    return ClaimArrays{A.st_p, A.st_s, A.wp_people, A.claim_p, A.claim_s, list_p, list_s, n_claimed};
}

// LDS queue of a contact block's successful draws.  A round of two slots
// adds at most 2 per thread; the queue is emptied when the next round might
// not fit, and after the last one.
constexpr int kPickRound = 2 * kContactThreads;
constexpr int kPickQueue = kPickRound + kContactThreads;
struct PickQueue {
    uint32_t n, errands, taken, base;
    uint32_t n_claim[2], claim_base[2];
    Pick at[kPickQueue];
    int32_t claimed[2][kPickQueue];
};

// A matrix row (row C: people per bucket).
__device__ __forceinline__ uint32_t* count_row(const CountTable& T, const CountRep& c, int row) {
    return T.pre + c.mbase + (int64_t)row * c.K;
}

// The chunk holding rank j of bucket b: the last c with pre[c][b] <= j
// (chunks without people of b share their successor's prefix).  People are
// spread evenly over the chunks, so the chunk is within C / (2 sqrt(total))
// (1 to 2) of j C / total: eight prefixes around it in one round trip nearly
// always hold it, else the window moves on.
__device__ __forceinline__ int chunk_of(const CountTable& T, const CountRep& c, uint32_t b, uint32_t j, uint32_t total,
                                        uint32_t& before, uint32_t& len) {
    constexpr int W = 8;
    const uint32_t* col = T.pre + c.mbase + b;
    int w = (int)((float)j * (float)c.C / (float)total) - W / 2 + 1;
    for (;;) {
        w = max(0, min(w, c.C - W + 1));  // rows w .. w + W - 1 of the C + 1 (row C: the total)
        uint32_t p[W];
#pragma unroll
        for (int i = 0; i < W; ++i) p[i] = col[(int64_t)min(w + i, c.C) * c.K];
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

// Marks (chunk, bucket) for collection.
__device__ __forceinline__ void mark_chunk(const CountTable& T, const CountRep& c, int chunk, uint32_t b,
                                           int32_t stamp) {
    atomicOr(T.marks + c.qbase + (int64_t)chunk * c.qw + (b >> 5), 1u << (b & 31));
    T.chunk_day[c.chunk0 + chunk] = stamp;
}

// A queued pick: finds and marks its chunk (and the next rank's, should the
// infector itself sit at this rank: only possible in its own chunk) and
// appends the pick to the day's list.
__device__ __forceinline__ void locate_pick(const CountTable& T, const Pick& p, uint32_t i, int day) {
    const CountRep c = T.reps[p.r];
    const uint32_t total = count_row(T, c, c.C)[p.at];
    uint32_t before, len;
    const int chunk = chunk_of(T, c, p.at, p.rank, total, before, len);
    mark_chunk(T, c, chunk, p.at, day + 1);
    T.pk_bucket[i] = p.at;
    T.pk_want[i] = p.rank - before;
    T.pk_claim[i] = p.claim;
    T.pk_payload[i] = p.payload;
    T.pk_idx[i] = p.idx;
    T.pk_r[i] = p.r;
    T.pk_chunk[i] = chunk;
    T.pk_len[i] = (int32_t)len;
    if (chunk == p.idx / c.A) {
        const uint32_t next = p.rank + 1 == total ? 0u : p.rank + 1;
        if (next < before || next >= before + len) {
            const int c2 = chunk_of(T, c, p.at, next, total, before, len);
            mark_chunk(T, c, c2, p.at, day + 1);
        }
    }
}

// Lists the infectors of a block's turn that are kept (all threads call).
__device__ __forceinline__ void list_infectors(const CountTable& T, bool keep, int32_t idx, int32_t pos, uint32_t f,
                                               int32_t r, bool with_r) {
    __shared__ uint32_t s_n, s_base;
    const int lane = threadIdx.x & 63;
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    const uint64_t m = __ballot(keep);
    uint32_t at = 0;
    if (lane == 0 && m) at = atomicAdd(&s_n, (uint32_t)__popcll(m));
    at = __shfl(at, 0, 64) + (uint32_t)__popcll(m & ((1ull << lane) - 1));
    __syncthreads();
    if (threadIdx.x == 0 && s_n) s_base = atomicAdd(&T.n[1], s_n);
    __syncthreads();
    if (keep) {
        const uint32_t i = s_base + at;
        T.sv_idx[i] = idx;
        T.sv_pos[i] = pos;
        T.sv_f[i] = f;
        if (with_r) T.sv_r[i] = r;
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
    for (uint32_t i0 = 0; i0 < n; i0 += blockDim.x) {
        const uint32_t i = i0 + tid;
        bool newp = false, news = false;
        int64_t slot = 0;
        if (i < n) {
            const Pick p = q.at[i];
            const uint32_t kind = p.payload >> 26;
            if (kind == 0) {
                locate_pick(T, p, q.base + atomicAdd(&q.taken, 1u), sts[p.r].day);
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
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        int32_t* list = k ? C.list_s : C.list_p;
        for (uint32_t i = tid; i < q.n_claim[k]; i += blockDim.x) list[q.claim_base[k] + i] = q.claimed[k][i];
    }
    __syncthreads();
    if (tid == 0) q.n = q.errands = q.taken = q.n_claim[0] = q.n_claim[1] = 0;
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
    __device__ __forceinline__ void round(bool last) const {
        __syncthreads();
        const uint32_t n = q->n;
        if (n && (last || n > (uint32_t)(kPickQueue - kPickRound))) flush_picks(T, C, *q, sts);
        __syncthreads();
    }
};

namespace {

// Keys and counts of a chunk.  VALU bound (the errand draws); the LDS adds,
// the 4-byte coalesced key stores and the row flush hide behind them.
template <bool WEEKEND>
__global__ __launch_bounds__(1024) void k_count(const int32_t* __restrict__ done, DayState* __restrict__ sts,
                                                const Model* __restrict__ models, const uint8_t* __restrict__ ages,
                                                CountTable T) {
    if (*done) return;
    extern __shared__ uint32_t s_cnt[];
    const CountBlock blk = T.chunks[blockIdx.x];
    DayState* st = sts + blk.r;
    if (st->done) return;
    const Model& M = models[blk.r];
    const CountRep c = T.reps[blk.r];
    const int tid = threadIdx.x, nt = blockDim.x;
    const uint32_t K = (uint32_t)c.K;
    for (int i = tid; i < c.K; i += nt) s_cnt[i] = 0;
    __syncthreads();
    const int64_t N = M.N;
    const int64_t a0 = (int64_t)blk.at * c.A, a1 = min(N, a0 + c.A);  // even a0
    const uint64_t eoff = st->rand_offset;  // the day's errand offset: it moves at the day's end
    bool bad = false;
    auto add = [&](uint32_t k) {
        if (k < K)
            atomicAdd(&s_cnt[k], 1u);
        else
            bad = true;
    };
    if (WEEKEND) {
        const ErrandWalk wk = pinned(M.we_walk);
        const int base = M.we_base, E = M.we_E;
        uint16_t* out = T.keys + c.abase;
        for (int64_t p = a0 + tid; p < a1; p += nt) {
            int32_t hour[3], loc[3];
            weekend_errands(M, wk, eoff + (uint64_t)(int64_t)(2 * (int32_t)p), hour, loc);
#pragma unroll
            for (int e = 0; e < 3; ++e) {
                const uint32_t k = (uint32_t)(hour[e] * E + (loc[e] - base));
                out[e * T.slots + p] = (uint16_t)k;
                add(k);
            }
        }
    } else {
        const ErrandWalk wk = pinned(M.wd_walk);
        const int base = M.wd_base, base1 = M.wd_base1 - M.wd_E;  // hour-1 keys follow the wd_E hour-0 keys
        const uint8_t* age = ages + c.abase;
        uint32_t* out0 = reinterpret_cast<uint32_t*>(T.keys + c.abase);
        uint32_t* out1 = reinterpret_cast<uint32_t*>(T.keys + T.slots + c.abase);
        for (int64_t g = a0 / 2 + tid; 2 * g < a1; g += nt) {
            const U4 u = draw4(eoff + (uint64_t)g, M.key0, M.key1);
            uint32_t w0 = 0, w1 = 0;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int64_t p = 2 * g + k;
                uint32_t k0 = kNoKey, k1 = kNoKey;
                if (p < a1) {
                    const bool adult = age[p] == kAgeAdult;
                    int32_t d1, d2;
                    weekday_dests(M, wk, u.w[2 * k], u.w[2 * k + 1], adult, d1, d2);
                    k0 = (uint32_t)(d1 - base);
                    add(k0);
                    if (adult) {
                        k1 = (uint32_t)(d2 - base1);
                        add(k1);
                    }
                }
                w0 |= (k0 & 0xFFFFu) << (16 * k);
                w1 |= (k1 & 0xFFFFu) << (16 * k);
            }
            out0[g] = w0;
            out1[g] = w1;
        }
    }
    if (bad) st->fault = 1;
    __syncthreads();
    uint32_t* row = T.pre + c.mbase + (int64_t)blk.at * c.K;
    for (int i = tid; i < c.K; i += nt) row[i] = s_cnt[i];
}

// Column prefixes of the count matrices, 64 buckets per block: 16 row groups
// sum up to 16 rows each in registers, so 256 rows take one round trip.
// Also clears the day's marks, picks and lists.
constexpr int kScanCols = 64, kScanGroups = 16, kScanRows = 16;
__global__ __launch_bounds__(kScanCols* kScanGroups) void k_count_scan(const int32_t* __restrict__ done,
                                                                       const DayState* __restrict__ sts,
                                                                       CountTable T) {
    if (*done) return;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < T.mark_words;
         i += (int64_t)gridDim.x * blockDim.x)
        T.marks[i] = 0u;
    if (blockIdx.x == 0 && threadIdx.x < 2) T.n[threadIdx.x] = 0u;
    const CountBlock blk = T.scans[blockIdx.x];
    if (sts[blk.r].done) return;
    const CountRep c = T.reps[blk.r];
    __shared__ uint32_t s_sum[kScanGroups][kScanCols];
    const int col = threadIdx.x % kScanCols, grp = threadIdx.x / kScanCols;
    const int b = blk.at + col;
    uint32_t* m = T.pre + c.mbase + b;
    uint32_t carry = 0;
    for (int s0 = 0; s0 < c.C; s0 += kScanGroups * kScanRows) {
        const int rows = min(c.C - s0, kScanGroups * kScanRows);
        const int per = (rows + kScanGroups - 1) / kScanGroups;
        const int r0 = s0 + grp * per, r1 = min(s0 + rows, r0 + per);
        uint32_t v[kScanRows], sum = 0;
#pragma unroll
        for (int i = 0; i < kScanRows; ++i) {
            v[i] = r0 + i < r1 && b < c.K ? m[(int64_t)(r0 + i) * c.K] : 0u;
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
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kScanRows; ++i) {
            if (r0 + i < r1 && b < c.K) m[(int64_t)(r0 + i) * c.K] = run;
            run += v[i];
        }
    }
    if (grp == 0 && b < c.K) m[(int64_t)c.C * c.K] = carry;
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
    uint32_t* start = T.cursor + c.mbase + (int64_t)blk.at * c.K;
    const uint32_t* row = count_row(T, c, blk.at);
    if (tid == 0) s_top = (uint32_t)(KPA * (c.abase + a0));
    for (int i = tid; i < c.K; i += nt) s_cur[i] = ~0u;
    __syncthreads();
    for (int i = tid; i < c.qw; i += nt) {
        uint32_t w = marks[i];
        while (w) {
            const int b = i * 32 + __ffs(w) - 1;
            w &= w - 1;
            start[b] = s_cur[b] = atomicAdd(&s_top, row[c.K + b] - row[b]);
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
        const int32_t* l = T.list + T.cursor[c.mbase + (int64_t)chunk * c.K + b];
        const int32_t v = rank_in_list(l, len, want, chunk * c.A, c.A, sub);
        if (v != idx || round) return v;
        const uint32_t total = count_row(T, c, c.C)[b];  // the next person instead (select_person)
        uint32_t j = count_row(T, c, chunk)[b] + want + 1, before;
        if (j == total) j = 0;
        chunk = chunk_of(T, c, b, j, total, before, len);
        want = j - before;
    }
}

__global__ __launch_bounds__(256) void k_resolve(DayState* __restrict__ g, CountTable T, ClaimArrays C) {
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
    int n_chunks = 0, n_scans = 0, threads = 0, kpa = 0;
    size_t lds = 0;
    int64_t entries = 0, mark_words = 0;
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
        lds = sizeof(uint32_t) * (size_t)kmax;
        threads = 1024;
        for (size_t r = 0; r < reps.size(); ++r) {
            CountRep& c = reps[r];
            c.A = count_chunk(N[r], c.K, kpa, std::max<int64_t>(1, want * N[r] / total));
            c.C = (int32_t)((N[r] + c.A - 1) / c.A);
            c.qw = (c.K + 31) / 32;
            c.mbase = entries;
            c.qbase = mark_words;
            c.chunk0 = (int32_t)chunks.size();
            entries += (int64_t)(c.C + 1) * c.K;
            mark_words += (int64_t)c.C * c.qw;
            for (int k = 0; k < c.C; ++k) chunks.push_back({(int32_t)r, k});
            for (int b = 0; b < c.K; b += kScanCols) scans.push_back({(int32_t)r, b});
        }
        n_chunks = (int)chunks.size();
        n_scans = (int)scans.size();
    }
    int upload(hipStream_t st) {
        if (!on) return 0;
        if (dev_alloc(&d_reps, (int64_t)reps.size()) || dev_alloc(&d_chunks, n_chunks) || dev_alloc(&d_scans, n_scans))
            return PT_ENOMEM;
        HIP_TRY(hipMemcpyAsync(d_reps, reps.data(), sizeof(CountRep) * reps.size(), hipMemcpyHostToDevice, st));
        HIP_TRY(hipMemcpyAsync(d_chunks, chunks.data(), sizeof(CountBlock) * n_chunks, hipMemcpyHostToDevice, st));
        HIP_TRY(hipMemcpyAsync(d_scans, scans.data(), sizeof(CountBlock) * n_scans, hipMemcpyHostToDevice, st));
        return 0;
    }
    void release() {
        dev_free(d_reps);
        dev_free(d_chunks);
        dev_free(d_scans);
        *this = CountPlan();
    }
};

// Buffers shared by the two layouts.
struct CountScratch {
    uint32_t *pre = nullptr, *cursor = nullptr, *marks = nullptr, *n = nullptr;
    int32_t* chunk_day = nullptr;
    int alloc(const CountPlan& a, const CountPlan& b) {
        const int64_t e = std::max(a.entries, b.entries);
        if (e == 0) return 0;
        return dev_alloc(&pre, e) || dev_alloc(&cursor, e) || dev_alloc(&marks, std::max(a.mark_words, b.mark_words)) ||
                       dev_alloc(&chunk_day, std::max(a.n_chunks, b.n_chunks)) || dev_alloc(&n, 2)
                   ? PT_ENOMEM
                   : 0;
    }
    void release() {
        dev_free(pre);
        dev_free(cursor);
        dev_free(marks);
        dev_free(chunk_day);
        dev_free(n);
    }
    void fill(CountTable& t, const CountPlan& p) const {
        t.reps = p.d_reps;
        t.chunks = p.d_chunks;
        t.scans = p.d_scans;
        t.pre = pre;
        t.cursor = cursor;
        t.marks = marks;
        t.mark_words = p.mark_words;
        t.chunk_day = chunk_day;
        t.n = n;
    }
};

// LDS above the default limit for the counting kernels.
inline hipError_t set_count_lds(const CountPlan& p) {
    if (!p.on || p.lds <= 64 * 1024) return hipSuccess;
    for (const void* k : {reinterpret_cast<const void*>(&k_count<false>), reinterpret_cast<const void*>(&k_count<true>),
                          reinterpret_cast<const void*>(&k_collect<false>),
                          reinterpret_cast<const void*>(&k_collect<true>)}) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(4 * kCountMaxK));
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Before contacts: keys, counts, prefixes.  After: lists, picks, claims.
inline void enqueue_counts(const CountPlan& p, const CountTable& t, const int32_t* done, DayState* sts,
                           const Model* models, const uint8_t* age, bool weekend, hipStream_t st, LaunchTimer* tm) {
    launch_lds(tm, weekend ? KC_GEN_WEEKEND : KC_GEN_WEEKDAY, weekend ? k_count<true> : k_count<false>,
               dim3(p.n_chunks), dim3(p.threads), p.lds, st, done, sts, models, age, t);
    launch(tm, KC_COUNT_SCAN, k_count_scan, dim3(p.n_scans), dim3(kScanCols * kScanGroups), st, done,
           (const DayState*)sts, t);
}

inline void enqueue_picks(const CountPlan& p, const CountTable& t, const ClaimArrays& c, DayState* g,
                          const DayState* sts, const Model* models, int grid, bool weekend, hipStream_t st,
                          LaunchTimer* tm) {
    launch_lds(tm, KC_COLLECT, weekend ? k_collect<true> : k_collect<false>, dim3(p.n_chunks), dim3(p.threads), p.lds,
               st, (const int32_t*)&g->done, sts, models, t);
    launch(tm, KC_RESOLVE, k_resolve, dim3(grid), dim3(256), st, g, t, c);
}

}  // namespace pt
