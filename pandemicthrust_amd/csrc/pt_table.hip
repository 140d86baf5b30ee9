// pt_table.hip — stand-alone location-table build on gfx950 (C ABI of
// pt_location_table, include/pandemic/pt_abi.h).
//
// A location table is what the reference builds each day with
// cub::DeviceRadixSort::SortPairs followed by thrust::lower_bound
// (PandemicSim.cu:1212-1248, :1316-1354, :3835-3862): the ids of the pairs
// grouped by bucket key, ascending within a key (the sort is stable and the
// ids come in ascending order), and offsets[k] = the number of keys below k.
// The build is the engine's own radix table build (pt_sort.hip).  Its radix
// scratch is one block of what the build's passes touch, and the block is
// kept for the next call: allocating and freeing 20 bytes per pair in six
// pieces took 10 of 11.5 ms for 20M pairs (freed device memory is cleared
// before it is handed out again, at some 40 GB/s).
#include <hip/hip_runtime.h>

#include <mutex>

#include "../../include/pandemic/pt_abi.h"
#include "pt_day.h"
#include "pt_sort.h"

using namespace pt;

namespace pt {

int location_table_args(const uint32_t* keys, int64_t n, int32_t n_buckets, const int32_t* people,
                        const int32_t* offsets) {
    if (n < 0 || n >= ((int64_t)1 << 31)) return fail(PT_EINVAL, "pair count %lld outside [0, 2^31)", (long long)n);
    if (n_buckets < 1 || n_buckets == 0x7FFFFFFF)
        return fail(PT_EINVAL, "bucket count %d outside [1, 2^31 - 1)", n_buckets);
    if (!offsets || (n > 0 && (!keys || !people))) return fail(PT_EINVAL, "null device pointer");
    return PT_OK;
}

namespace {

// One idle scratch block per device, of at most kKeepBytes.  A call takes the
// block out (calls that overlap allocate their own), waits for its stream, and
// puts its block back in place of a smaller one.  A block more than four times
// what a call needs is freed instead of used, every block is freed when an
// allocation of the library fails, and a caller may free it
// (pt_location_table_release).
constexpr size_t kKeepBytes = (size_t)512 << 20;
constexpr int kMaxDevices = 64;
struct Block {
    void* p = nullptr;
    size_t bytes = 0;
};
std::mutex g_mu;
Block g_idle[kMaxDevices];

Block take_block(int device) {
    Block b;
    if (device < 0 || device >= kMaxDevices) return b;
    std::lock_guard<std::mutex> lock(g_mu);
    std::swap(b, g_idle[device]);
    return b;
}

void put_block(int device, Block b) {
    if (device >= 0 && device < kMaxDevices && b.bytes <= kKeepBytes) {
        std::lock_guard<std::mutex> lock(g_mu);
        if (b.bytes > g_idle[device].bytes) std::swap(b, g_idle[device]);
    }
    if (b.p) (void)hipFree(b.p);
}

}  // namespace

hipError_t device_malloc(void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess) return e;
    bool gave = false;
    for (int d = 0; d < kMaxDevices; ++d) {
        const Block b = take_block(d);
        if (b.p) gave = hipFree(b.p) == hipSuccess || gave;
    }
    if (!gave) return e;
    (void)hipGetLastError();
    return hipMalloc(p, bytes);
}

}  // namespace pt

extern "C" int pt_location_table(const uint32_t* keys, int64_t n, int32_t n_buckets, int32_t* people,
                                 int32_t* offsets, int32_t device, void* stream) {
    if (int rc = location_table_args(keys, n, n_buckets, people, offsets)) return rc;
    DeviceScope ds(device);
    HIP_TRY(ds.err);
    hipStream_t st = (hipStream_t)stream;
    if (is_small_table(keys, n, n_buckets, people, offsets)) {
        hipError_t e = build_small_table(keys, n, n_buckets, people, offsets, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e != hipSuccess) return fail(PT_EDEVICE, "location table: %s", hipGetErrorString(e));
        return PT_OK;
    }
    const size_t need = table_scratch_bytes(n, n_buckets);
    Block block = take_block(device);
    if (block.bytes < need || block.bytes / 4 > need) {
        if (block.p) (void)hipFree(block.p);
        block = Block{nullptr, need};
        if (device_malloc(&block.p, need) != hipSuccess)
            return fail(PT_ENOMEM, "radix scratch for %lld pairs", (long long)n);
    }
    TableScratch ts;
    table_scratch_carve(ts, (unsigned char*)block.p, n, n_buckets);
    hipError_t e = build_table(ts, const_cast<uint32_t*>(keys), nullptr, n, nullptr, n_buckets, ID_IDENTITY,
                               (int32_t)n, people, offsets, nullptr, st, nullptr);
    if (e == hipSuccess) e = hipStreamSynchronize(st);  // the block is free for other streams from here
    if (e != hipSuccess) {
        (void)hipFree(block.p);
        return fail(PT_EDEVICE, "location table: %s", hipGetErrorString(e));
    }
    put_block(device, block);
    return PT_OK;
}

extern "C" int pt_location_table_release(int32_t device) {
    if (device < 0 || device >= kMaxDevices) return fail(PT_EINVAL, "device %d outside [0, %d)", device, kMaxDevices);
    DeviceScope ds(device);
    HIP_TRY(ds.err);
    const Block block = take_block(device);
    if (block.p) HIP_TRY(hipFree(block.p));
    return PT_OK;
}
