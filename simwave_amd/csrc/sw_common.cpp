// Process-wide state shared by the eight variant libraries.
//
// Each variant library (libsimwave_hip_<2|3>d_<cd|vd>_<f32|f64>.so) links
// against this one, so however the libraries are loaded (ctypes loads them
// RTLD_LOCAL) the dynamic loader maps a single copy per process and every
// variant sees the same counters.
//
// The receiver-overlap lease: a forward run or plan that puts the receiver
// gather on a second stream of its own (flag 4 of the device entries) joins
// the two streams with event waits in both directions.  Streams share the
// device's few hardware queues, and when several host threads enqueue such
// two-way waits at once, a wait can land in a queue ahead of the work it
// waits for, behind another stream's wait on that queue's work: a cycle
// that never drains.  One holder per process cannot form such a cycle, so
// the lease admits one holder at a time.
//
// The kept blocks: device memory that one gradient is done with, for the next
// (the variant libraries allocate and free it; here is only the list, oldest
// first).
#include <atomic>
#include <mutex>
#include <vector>

#define SW_COMMON_EXPORT extern "C" __attribute__((visibility("default")))

namespace {
std::atomic<int> g_overlap_holders{0};

struct KeptBlock {
    void *p;
    unsigned long long bytes;
    int device;
};
std::mutex g_blocks_mutex;
std::vector<KeptBlock> g_blocks;

unsigned long long kept_bytes(int device)
{
    unsigned long long sum = 0;
    for (const KeptBlock &b : g_blocks)
        if (b.device == device)
            sum += b.bytes;
    return sum;
}
}

// 1 if the caller now holds the lease, 0 if another run or plan holds it.
SW_COMMON_EXPORT int simwave_hip_overlap_acquire(void)
{
    int expected = 0;
    return g_overlap_holders.compare_exchange_strong(expected, 1) ? 1 : 0;
}

SW_COMMON_EXPORT void simwave_hip_overlap_release(void)
{
    g_overlap_holders.store(0);
}

// Current holders (0 or 1).
SW_COMMON_EXPORT int simwave_hip_overlap_holders(void)
{
    return g_overlap_holders.load();
}

// Bytes that `device` holds in kept blocks.
SW_COMMON_EXPORT unsigned long long simwave_hip_block_held(int device)
{
    std::lock_guard<std::mutex> g(g_blocks_mutex);
    return kept_bytes(device);
}

// The smallest kept block of `device` that holds `bytes` and is at most a
// quarter larger, taken off the list (its size in *got), or null.
SW_COMMON_EXPORT void *simwave_hip_block_take(int device, unsigned long long bytes,
                                              unsigned long long *got)
{
    std::lock_guard<std::mutex> g(g_blocks_mutex);
    size_t best = g_blocks.size();
    for (size_t i = 0; i < g_blocks.size(); i++) {
        const KeptBlock &b = g_blocks[i];
        if (b.device == device && b.bytes >= bytes && b.bytes - bytes <= bytes / 4 &&
            (best == g_blocks.size() || b.bytes < g_blocks[best].bytes))
            best = i;
    }
    if (best == g_blocks.size())
        return nullptr;
    void *p = g_blocks[best].p;
    *got = g_blocks[best].bytes;
    g_blocks.erase(g_blocks.begin() + (long)best);
    return p;
}

// Keeps a block nothing uses any more if `device` then holds at most `limit`
// bytes: 1, or 0 where the caller has to free it.
SW_COMMON_EXPORT int simwave_hip_block_put(int device, void *p, unsigned long long bytes,
                                           unsigned long long limit)
{
    std::lock_guard<std::mutex> g(g_blocks_mutex);
    if (bytes > limit || kept_bytes(device) > limit - bytes)
        return 0;
    try {
        g_blocks.push_back({p, bytes, device});
    } catch (...) {
        return 0;
    }
    return 1;
}

// The oldest kept block of `device`, taken off the list for the caller to
// free, while the device holds more than `limit` bytes; otherwise null.
SW_COMMON_EXPORT void *simwave_hip_block_evict(int device, unsigned long long limit)
{
    std::lock_guard<std::mutex> g(g_blocks_mutex);
    if (kept_bytes(device) <= limit)
        return nullptr;
    for (size_t i = 0; i < g_blocks.size(); i++)
        if (g_blocks[i].device == device) {
            void *p = g_blocks[i].p;
            g_blocks.erase(g_blocks.begin() + (long)i);
            return p;
        }
    return nullptr;
}
