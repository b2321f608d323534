// The idle work blocks of the solvers (WorkArray, internal.hpp) and the
// allocations that give them back before they fail.  Host code over the
// runtime's allocation calls alone, so its rules are tested on the host against
// a model of those calls.

#include <cstring>

#include "internal.hpp"

namespace sbh {

namespace {

struct WorkPool {
    std::mutex mu;
    std::vector<WorkBlock> idle;  // oldest first, never more than reserved here
    size_t bytes[2] = {0, 0};     // device memory, pinned host memory
    WorkPool() { idle.reserve(WORK_IDLE_BLOCKS); }

    // Takes block i out; the lock is held.
    WorkBlock take(size_t i) {
        const WorkBlock b = idle[i];
        idle.erase(idle.begin() + (std::ptrdiff_t)i);
        bytes[b.pinned] -= b.bytes;
        return b;
    }
};

// never destroyed: arrays may outlive the library's static objects
WorkPool& work_pool() {
    static WorkPool* pool = new WorkPool;
    return *pool;
}

void work_free(const WorkBlock& b) {
    if (b.pinned)
        (void)hipHostFree(b.ptr);
    else
        (void)hipFree(b.ptr);
}

size_t idle_limit(bool pinned) { return pinned ? WORK_IDLE_PINNED_LIMIT : WORK_IDLE_LIMIT; }

// One more try after the idle blocks, of both kinds, are given back
template <typename Alloc>
void* with_trim(Alloc&& alloc) {
    void* p = nullptr;
    hipError_t e = alloc(&p);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();  // clear it
        work_trim();
        e = alloc(&p);
    }
    SBH_HIP(e);
    return p;
}

}  // namespace

IdleBytes work_trim() {
    WorkPool& pool = work_pool();
    IdleBytes freed;
    for (;;) {
        WorkBlock b;
        {
            std::lock_guard<std::mutex> lk(pool.mu);
            if (pool.idle.empty()) return freed;
            b = pool.take(pool.idle.size() - 1);
        }
        (b.pinned ? freed.pinned : freed.device) += (int64_t)b.bytes;
        work_free(b);
    }
}

int64_t work_idle_bytes(int device) {
    WorkPool& pool = work_pool();
    std::lock_guard<std::mutex> lk(pool.mu);
    int64_t sum = 0;
    for (const WorkBlock& b : pool.idle)
        if (!b.pinned && b.device == device) sum += (int64_t)b.bytes;
    return sum;
}

int64_t work_fill(int byte) {
    WorkPool& pool = work_pool();
    std::lock_guard<std::mutex> lk(pool.mu);
    int64_t sum = 0;
    for (const WorkBlock& b : pool.idle) {
        if (b.pinned)
            std::memset(b.ptr, byte, b.bytes);
        else
            SBH_HIP(hipMemset(b.ptr, byte, b.bytes));
        sum += (int64_t)b.bytes;
    }
    SBH_HIP(hipDeviceSynchronize());
    return sum;
}

void* device_malloc(size_t bytes) {
    return with_trim([&](void** p) { return hipMalloc(p, bytes); });
}

void* pinned_malloc(size_t bytes) {
    return with_trim([&](void** p) { return hipHostMalloc(p, bytes, hipHostMallocDefault); });
}

WorkBlock work_take(size_t bytes, bool pinned) {
    WorkBlock b;
    b.bytes = (bytes + 255) / 256 * 256;
    b.pinned = pinned;
    SBH_HIP(hipGetDevice(&b.device));
    {
        // the smallest idle block that fits without wasting more than a quarter
        WorkPool& pool = work_pool();
        std::lock_guard<std::mutex> lk(pool.mu);
        size_t best = pool.idle.size();
        for (size_t i = 0; i < pool.idle.size(); ++i) {
            const WorkBlock& c = pool.idle[i];
            if (c.device == b.device && c.pinned == pinned && c.bytes >= b.bytes &&
                c.bytes <= b.bytes + b.bytes / 4 + 65536 && (best == pool.idle.size() || c.bytes < pool.idle[best].bytes))
                best = i;
        }
        if (best < pool.idle.size()) return pool.take(best);
    }
    b.ptr = pinned ? pinned_malloc(b.bytes) : device_malloc(b.bytes);
    return b;
}

void work_give(const WorkBlock& b) {
    // hipFree's order: nothing on the device uses the block any more, whatever
    // stream it was on
    int device = -1;
    if (b.bytes > std::min(WORK_BLOCK_LIMIT, idle_limit(b.pinned)) || hipGetDevice(&device) != hipSuccess ||
        device != b.device || hipDeviceSynchronize() != hipSuccess) {
        work_free(b);
        return;
    }
    WorkPool& pool = work_pool();
    for (;;) {
        WorkBlock oldest;
        {
            std::lock_guard<std::mutex> lk(pool.mu);
            size_t out = 0;
            if (pool.bytes[b.pinned] + b.bytes > idle_limit(b.pinned)) {
                while (pool.idle[out].pinned != b.pinned) ++out;  // there is one: b alone is within the limit
            } else if (pool.idle.size() < WORK_IDLE_BLOCKS) {
                pool.idle.push_back(b);
                pool.bytes[b.pinned] += b.bytes;
                return;
            }
            oldest = pool.take(out);
        }
        work_free(oldest);
    }
}

}  // namespace sbh
