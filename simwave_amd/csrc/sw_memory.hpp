// Device memory of one run: the arena that every entry point allocates from,
// over the memory calls of `Api` (the HIP runtime's in the libraries).
//
// Host code only, with no HIP type in it, so that what happens when the
// device runs out of memory can be tested without one.
#pragma once
#include <algorithm>
#include <cstddef>
#include <vector>

namespace sw {

// At most this many bytes per device are kept from one gradient for the next.
constexpr size_t kKeptBlockBytes = (size_t)8 << 30;

// Frees the oldest kept blocks of `device` on `st` until at most `limit`
// bytes are left.
template <typename Api>
void drop_blocks(int device, size_t limit, typename Api::stream st)
{
    while (void *p = Api::evict(device, limit))
        Api::free(p, st);
}

// Stream-ordered device allocations released when the object dies.  With a
// base pointer it instead hands out consecutive 256-byte aligned pieces of
// that caller-owned region (no allocation, nothing to free) and fails once
// `cap` bytes are used.
template <typename Api>
struct Arena {
    typedef typename Api::stream Stream;
    Stream stream;
    std::vector<void *> ptrs;
    char *base = nullptr;
    size_t cap = 0, used = 0;
    // Blocks kept from one run for the next (keep_blocks): the run's own list,
    // those it released on the way free for its later requests (one stream, so
    // in order).
    struct Block {
        void *p;
        size_t bytes;
        bool free;
    };
    int keep_device = -1;
    std::vector<Block> blocks;
    // bytes requested so far, and the most of them that the run may (0: any)
    size_t requested = 0;
    const size_t limit = Api::limit();

    explicit Arena(Stream s) : stream(s) {}
    Arena(Stream s, void *region, size_t bytes)
        : stream(s), base(static_cast<char *>(region)), cap(bytes)
    {
    }
    Arena(const Arena &) = delete;
    Arena &operator=(const Arena &) = delete;
    ~Arena()
    {
        for (void *p : ptrs)
            Api::free(p, stream);
        // kept blocks may serve any stream next: only once this one is done
        const bool done = Api::synchronize(stream);
        for (const Block &b : blocks) {
            if (done && b.bytes <= kKeptBlockBytes) {
                drop_blocks<Api>(keep_device, kKeptBlockBytes - b.bytes, stream);
                if (Api::put(keep_device, b.p, b.bytes, kKeptBlockBytes))
                    continue;
            }
            Api::free(b.p, stream);
        }
    }

    // From here on requests of kKeepMin bytes and more are served from blocks
    // that outlive the run: the runtime's stream-ordered allocations and frees
    // map and unmap memory, 30 us and up to 3 ms each on the host (a gradient
    // of 200 x 220 x 240 points spent 4.4 of its 16.4 ms so).  The oldest kept
    // blocks go first, and simwave_hip_trim_pool, or an allocation that finds
    // the device full, gives all of them back.
    static constexpr size_t kKeepMin = (size_t)1 << 20;
    void keep_blocks() { keep_device = Api::device(); }

    // `bytes` of fresh memory on `st`.  Where the device has none left, the
    // kept blocks and whatever freed memory the pool holds go back to it first
    // (on `device`, the current one if negative).
    static void *fresh(size_t bytes, Stream st, Arena *own = nullptr)
    {
        void *p = nullptr;
        if (Api::alloc(&p, bytes, st))
            return p;
        if (own)
            own->free_released();
        drop_blocks<Api>(Api::device(), 0, st);
        // the frees above are stream-ordered: the pool can only give back
        // what the stream has passed
        Api::synchronize(st);
        Api::trim();
        if (!Api::alloc(&p, bytes, st))
            Api::out_of_memory(bytes);
        return p;
    }

    template <typename T>
    T *alloc(size_t count)
    {
        if (count == 0)
            return nullptr;
        const size_t bytes = count * sizeof(T);
        if (base) {
            const size_t whole = (bytes + 255) / 256 * 256;
            if (whole > cap - used)
                Api::region_full(bytes, cap, used);
            void *p = base + used;
            used += whole;
            return static_cast<T *>(p);
        }
        requested += bytes;
        if (limit && requested > limit)
            Api::out_of_memory(bytes);
        if (keep_device >= 0 && bytes >= kKeepMin)
            return static_cast<T *>(alloc_block(bytes));
        ptrs.reserve(ptrs.size() + 1);
        void *p = fresh(bytes, stream, this);
        ptrs.push_back(p);
        return static_cast<T *>(p);
    }

    void release(void *p)
    {
        for (Block &b : blocks)
            if (b.p == p) {
                b.free = true;
                return;
            }
        auto it = std::find(ptrs.begin(), ptrs.end(), p);
        if (it != ptrs.end()) {
            Api::free(p, stream);
            ptrs.erase(it);
        }
    }

private:
    void *alloc_block(size_t bytes)
    {
        for (Block &b : blocks)
            if (b.free && b.bytes >= bytes && b.bytes - bytes <= bytes / 4) {
                b.free = false;
                return b.p;
            }
        blocks.reserve(blocks.size() + 1);
        size_t got = bytes;
        void *p = Api::take(keep_device, bytes, &got);
        if (!p) {
            got = bytes;
            p = fresh(bytes, stream, this);
        }
        blocks.push_back({p, got, false});
        return p;
    }

    // The blocks this run has released, back to the device.
    void free_released()
    {
        for (size_t i = blocks.size(); i-- > 0;)
            if (blocks[i].free) {
                Api::free(blocks[i].p, stream);
                blocks.erase(blocks.begin() + (std::ptrdiff_t)i);
            }
    }
};

}  // namespace sw
