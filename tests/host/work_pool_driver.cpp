// Runs sonium_amd/csrc/work_pool.cpp against a model of the runtime's
// allocation calls: one memory of `capacity` bytes for both kinds, and the
// blocks live in it.  Prints the failed checks; the exit status is their number.

#include <cstdio>
#include <cstdlib>
#include <map>
#include <thread>

#include "internal.hpp"

namespace {
std::mutex mu;
std::map<void*, std::pair<size_t, bool>> live;  // block -> bytes, pinned
size_t capacity = ~(size_t)0, used = 0;
uintptr_t next_address = 4096;
int failures = 0;

hipError_t model_malloc(void** p, size_t bytes, bool pinned) {
    std::lock_guard<std::mutex> lk(mu);
    if (used + bytes > capacity) return hipErrorOutOfMemory;
    *p = reinterpret_cast<void*>(next_address);
    next_address += bytes + 4096;
    live[*p] = {bytes, pinned};
    used += bytes;
    return hipSuccess;
}
hipError_t model_free(void* p, bool pinned) {
    std::lock_guard<std::mutex> lk(mu);
    auto it = live.find(p);
    if (it == live.end() || it->second.second != pinned) {
        std::printf("a block freed twice or as the other kind\n");
        ++failures;
        return hipErrorInvalidValue;
    }
    used -= it->second.first;
    live.erase(it);
    return hipSuccess;
}
size_t held(bool pinned) {
    std::lock_guard<std::mutex> lk(mu);
    size_t sum = 0;
    for (auto& b : live)
        if (b.second.second == pinned) sum += b.second.first;
    return sum;
}
void check(bool ok, const char* what) {
    if (ok) return;
    std::printf("failed: %s\n", what);
    ++failures;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) { return model_malloc(p, bytes, false); }
hipError_t hipFree(void* p) { return model_free(p, false); }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { return model_malloc(p, bytes, true); }
hipError_t hipHostFree(void* p) { return model_free(p, true); }
hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "out of memory"; }
}

using namespace sbh;

int main() {
    constexpr size_t MB = (size_t)1 << 20;
    // a block comes back for the same size, not for one that would waste it
    WorkBlock a = work_take(8 * MB, false);
    void* first = a.ptr;
    work_give(a);
    a = work_take(7 * MB, false);
    check(a.ptr == first, "reuse");
    work_give(a);
    a = work_take(2 * MB, false);
    check(a.ptr != first, "no reuse for a quarter of the size");
    WorkBlock p = work_take(8 * MB, true);
    check(p.ptr != first && p.pinned, "kinds apart");
    work_give(a);
    work_give(p);
    // idle memory of each kind within its limit, whatever is given back
    std::vector<WorkBlock> blocks;
    for (int i = 0; i < 100; ++i) blocks.push_back(work_take((1 + i % 7) * 4 * MB, true));
    for (int i = 0; i < 40; ++i) blocks.push_back(work_take(300 * MB, false));
    for (const WorkBlock& b : blocks) work_give(b);
    check(held(true) <= WORK_IDLE_PINNED_LIMIT && held(true) > 0, "pinned limit");
    check(held(false) <= WORK_IDLE_LIMIT && held(false) > 0, "device limit");
    blocks.clear();
    for (int i = 0; i < 300; ++i) blocks.push_back(work_take(256, i & 1));
    for (const WorkBlock& b : blocks) work_give(b);
    check(live.size() <= WORK_IDLE_BLOCKS, "number of blocks");
    const WorkBlock big = work_take(WORK_IDLE_PINNED_LIMIT + 1, true);
    work_give(big);
    check(live.find(big.ptr) == live.end(), "a pinned block above the limit is not kept");
    const size_t device = held(false), pinned = held(true);
    check(work_idle_bytes(0) == (int64_t)device && work_idle_bytes(1) == 0, "idle bytes of a device");
    const IdleBytes freed = work_trim();
    check(live.empty() && work_idle_bytes(0) == 0, "trim");
    check(freed.device == (int64_t)device && freed.pinned == (int64_t)pinned, "bytes given back");
    // an allocation of either kind that finds the memory full of idle blocks
    capacity = 100 * MB;
    for (bool pinned : {false, true}) {
        work_give(work_take(90 * MB, false));
        try {
            const WorkBlock b = work_take(50 * MB, pinned);
            check(held(!pinned) == 0 && used == b.bytes, "the idle block made room");
            work_give(b);
        } catch (const Error&) {
            check(false, "an allocation failed while idle blocks held the memory");
        }
        work_trim();
    }
    work_give(work_take(90 * MB, false));
    void* q = nullptr;
    try {
        q = pinned_malloc(60 * MB);
        check(held(false) == 0, "pinned_malloc made room");
        (void)hipHostFree(q);
    } catch (const Error&) {
        check(false, "pinned_malloc failed while idle blocks held the memory");
    }
    try {
        (void)device_malloc(200 * MB);
        check(false, "more than there is");
    } catch (const Error& e) {
        check(e.code == SBH_ERR_OUT_OF_MEMORY, "out of memory is typed");
    }
    capacity = ~(size_t)0;
    // threads that exchange blocks: each block has one owner
    std::vector<std::thread> threads;
    for (int t = 0; t < 8; ++t)
        threads.emplace_back([t] {
            for (int i = 0; i < 2000; ++i) {
                WorkBlock x = work_take((1 + (i * 7 + t) % 13) * 65536, i & 1), y = work_take(1 << 20, false);
                if (i % 97 == 0) work_trim();
                work_give(y);
                work_give(x);
            }
        });
    for (auto& t : threads) t.join();
    check(held(true) <= WORK_IDLE_PINNED_LIMIT && live.size() <= WORK_IDLE_BLOCKS, "limits after the threads");
    work_trim();
    check(live.empty() && used == 0, "every block given back once");
    std::printf("%d failed checks\n", failures);
    return failures;
}
