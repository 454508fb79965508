// device_memory.hpp -- device memory of the library's calls and formats (host code only).
#pragma once
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstddef>
#include <mutex>
#include <new>
#include <utility>
#include <vector>

#include "hip_error.hpp"

namespace vcsrmc {

// hipMalloc for everything the library allocates: where memory is short, once more after the kept
// blocks and this call's unused ones went back.  On failure the runtime's error is cleared, so a
// later launch does not report it.
inline hipError_t device_malloc(void** p, size_t bytes);

// ---- device memory owned for the duration of a scope ----------------------------------
template <typename T>
struct DevBuf {
    T* p = nullptr;
    size_t n = 0;
    DevBuf() = default;
    explicit DevBuf(size_t count) { alloc(count); }
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    DevBuf(DevBuf&& o) noexcept : p(o.p), n(o.n) { o.p = nullptr; o.n = 0; }
    DevBuf& operator=(DevBuf&& o) noexcept {
        if (this != &o) { release(); p = o.p; n = o.n; o.p = nullptr; o.n = 0; }
        return *this;
    }
    ~DevBuf() { release(); }
    // On failure the buffer stays empty (p null, n 0) and the runtime's error is cleared, so
    // a later launch does not report it.
    void alloc(size_t count) {
        release();
        if (!count) return;
        const hipError_t e = device_malloc((void**)&p, count * sizeof(T));
        if (e != hipSuccess) {
            p = nullptr;
            throw_hip(e, "hipMalloc", __FILE__, __LINE__);
        }
        n = count;
    }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    T* take() { T* q = p; p = nullptr; n = 0; return q; }
};

// ---- scratch of one call ----------------------------------------------------------------
// Temporaries of one library call come from an arena that lives as long as the call: a few large
// device blocks, handed out and taken back on the host.  Everything a call enqueues goes to its
// one stream, so a block taken back may be handed out again at once: the next kernels that write
// it follow the ones that read it.  A hipMalloc and hipFree for each of the ~460 temporaries of a
// format build instead cost the 27-point stencil 100^3 about 30 of its 68 ms.
//
// The blocks of a call that has waited for its stream go to a cache for later calls, on any thread
// or stream: the driver clears memory that is freed, and a program that builds or orders one matrix
// after another frees faster than that (builds of the stencil in a row: 14 ms at first, 34 once no
// cleared memory is left; orderings of a 64^3 mesh 3.6, then 17).  The cache holds at most
// kMaxBytes, gives back a block that the last kIdleCalls calls with scratch did not take, and all of
// them when any allocation of the library finds memory short (device_malloc) or the caller asks for it
// (vcsrmc_release_scratch): a program that builds once and then multiplies makes no later call that
// would give them back.  A call that ends in an error frees its blocks (hipFree waits for the device).
class BlockCache {
public:
    static BlockCache& instance() {
        static BlockCache* c = new BlockCache;  // not destroyed: the runtime may be gone by then
        return *c;
    }
    // The smallest kept block of at least `bytes` on the device, or null.
    char* take(int device, size_t bytes, size_t& size) {
        std::lock_guard<std::mutex> lock(m_);
        size_t best = kept_.size();
        for (size_t i = 0; i < kept_.size(); ++i)
            if (kept_[i].device == device && kept_[i].size >= bytes &&
                (best == kept_.size() || kept_[i].size < kept_[best].size))
                best = i;
        if (best == kept_.size()) return nullptr;
        char* p = kept_[best].p;
        size = kept_[best].size;
        total_ -= size;
        kept_.erase(kept_.begin() + best);
        return p;
    }
    // The blocks of one call.
    void give(int device, const std::vector<std::pair<char*, size_t>>& blocks) noexcept {
        std::vector<char*> out;
        try {
            std::lock_guard<std::mutex> lock(m_);
            out.reserve(kept_.size() + blocks.size());
            kept_.reserve(kept_.size() + blocks.size());
            ++calls_;
            for (const auto& [p, size] : blocks) {
                kept_.push_back(Kept{device, p, size, calls_});
                total_ += size;
            }
            for (size_t i = 0; i < kept_.size();)  // oldest first
                if (total_ > kMaxBytes || calls_ - kept_[i].call > kIdleCalls) {
                    out.push_back(kept_[i].p);
                    total_ -= kept_[i].size;
                    kept_.erase(kept_.begin() + i);
                } else {
                    ++i;
                }
        } catch (const std::bad_alloc&) {  // of the two reserves: nothing was kept
            for (const auto& b : blocks) (void)hipFree(b.first);
        }
        for (char* q : out) (void)hipFree(q);
    }
    size_t kept(int device) {
        std::lock_guard<std::mutex> lock(m_);
        size_t bytes = 0;
        for (const Kept& k : kept_) bytes += k.device == device ? k.size : 0;
        return bytes;
    }
    // Whether there were any.
    bool give_back_all() {
        std::vector<Kept> out;
        {
            std::lock_guard<std::mutex> lock(m_);
            out.swap(kept_);
            total_ = 0;
        }
        for (const Kept& k : out) (void)hipFree(k.p);
        return !out.empty();
    }

private:
    static constexpr size_t kMaxBytes = (size_t)2 << 30;
    static constexpr unsigned long long kIdleCalls = 16;
    struct Kept {
        int device;
        char* p;
        size_t size;
        unsigned long long call;
    };
    std::mutex m_;
    std::vector<Kept> kept_;
    size_t total_ = 0;
    unsigned long long calls_ = 0;
};

class Arena {
public:
    Arena() = default;
    Arena(const Arena&) = delete;
    Arena& operator=(const Arena&) = delete;
    ~Arena() {
        if (idle_ && !blocks_.empty()) {
            try {
                std::vector<std::pair<char*, size_t>> all;
                for (const Block& b : blocks_) all.emplace_back(b.p, b.size);
                BlockCache::instance().give(device_, all);
                return;
            } catch (const std::bad_alloc&) {
            }
        }
        for (Block& b : blocks_) (void)hipFree(b.p);
    }
    // The call has waited for its stream: nothing on the device uses the blocks any more.
    void idle() { idle_ = true; }
    // The size of the first block (0: as large as what asks for it); later ones are as large as what
    // asks for them, or kBlock.  A large one is not reserved ahead unless four times as much is
    // free: what a call makes to last, a format, has to find room beside it.
    void reserve(size_t bytes) {
        first_ = bytes ? std::max(bytes, kBlock) : 0;
        if (first_ > kLargeReserve && first_ > available() / 4) first_ = kBlock;
    }
    // Free memory of the current device for temporaries of this call: the driver's, what is kept from
    // earlier calls, and what this call holds and does not use.
    size_t available() {
        int device = 0;
        size_t bytes = 0, total = 0;
        if (hipGetDevice(&device) != hipSuccess || hipMemGetInfo(&bytes, &total) != hipSuccess) {
            (void)hipGetLastError();
            return 0;
        }
        bytes += BlockCache::instance().kept(device);
        for (const Block& b : blocks_)
            for (const Range& r : b.free) bytes += r.size;
        return bytes;
    }
    void* take(size_t bytes) {
        bytes = (bytes + kAlign - 1) / kAlign * kAlign;
        for (Block& b : blocks_)
            for (size_t i = 0; i < b.free.size(); ++i) {
                Range& r = b.free[i];
                if (r.size < bytes) continue;
                void* p = b.p + r.at;
                r.at += bytes;
                r.size -= bytes;
                if (r.size == 0) b.free.erase(b.free.begin() + i);
                return p;
            }
        size_t size = std::max(bytes, blocks_.empty() ? first_ : kBlock);
        blocks_.reserve(blocks_.size() + 1);
        if (device_ < 0) VCSRMC_HIP(hipGetDevice(&device_));
        char* p = BlockCache::instance().take(device_, size, size);
        hipError_t e = p ? hipSuccess : device_malloc((void**)&p, size);
        if (e == hipErrorOutOfMemory && size > bytes) {  // only what is asked for
            size = bytes;
            e = device_malloc((void**)&p, size);
        }
        if (e != hipSuccess) throw_hip(e, "hipMalloc", __FILE__, __LINE__);
        blocks_.push_back(Block{p, size, {}});
        if (size > bytes) blocks_.back().free.push_back(Range{bytes, size - bytes});
        return p;
    }
    void give(void* q, size_t bytes) {
        bytes = (bytes + kAlign - 1) / kAlign * kAlign;
        char* p = static_cast<char*>(q);
        for (Block& b : blocks_) {
            if (p < b.p || p >= b.p + b.size) continue;
            const size_t at = (size_t)(p - b.p);
            size_t i = 0;
            while (i < b.free.size() && b.free[i].at < at) ++i;
            b.free.insert(b.free.begin() + i, Range{at, bytes});
            if (i + 1 < b.free.size() && at + bytes == b.free[i + 1].at) {
                b.free[i].size += b.free[i + 1].size;
                b.free.erase(b.free.begin() + i + 1);
            }
            if (i > 0 && b.free[i - 1].at + b.free[i - 1].size == at) {
                b.free[i - 1].size += b.free[i].size;
                b.free.erase(b.free.begin() + i);
            }
            return;
        }
    }

    // Blocks of which nothing is in use go back to the driver; whether there were any.
    bool give_back_unused() {
        bool any = false;
        for (size_t i = 0; i < blocks_.size();) {
            Block& b = blocks_[i];
            if (b.free.size() == 1 && b.free[0].size == b.size) {
                if (!any) (void)hipDeviceSynchronize();  // kernels of this call may still use them
                (void)hipFree(b.p);
                blocks_.erase(blocks_.begin() + i);
                any = true;
            } else {
                ++i;
            }
        }
        return any;
    }

private:
    static constexpr size_t kAlign = 256, kBlock = (size_t)32 << 20, kLargeReserve = (size_t)1 << 30;
    struct Range {
        size_t at, size;
    };
    struct Block {
        char* p;
        size_t size;
        std::vector<Range> free;  // by offset, none touching the next
    };
    std::vector<Block> blocks_;
    size_t first_ = 0;
    int device_ = -1;
    bool idle_ = false;
};

// The arena of the call that runs on this thread: the outermost ScratchScope's.
inline thread_local Arena* tl_arena = nullptr;

inline hipError_t device_malloc(void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        const bool unused = tl_arena && tl_arena->give_back_unused();
        const bool kept = BlockCache::instance().give_back_all();
        if (unused || kept) e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) (void)hipGetLastError();
    return e;
}

struct ScratchScope {
    Arena own;
    const bool outer;
    explicit ScratchScope(size_t expected_bytes) : outer(tl_arena == nullptr) {
        if (!outer) return;
        own.reserve(expected_bytes);
        tl_arena = &own;
    }
    ~ScratchScope() {
        if (outer) tl_arena = nullptr;
    }
    // Called once the call has waited for its stream.
    void idle() { own.idle(); }
};

// A temporary of the current call: made and dropped inside a ScratchScope of its thread.
template <typename T>
struct TmpBuf {
    T* p = nullptr;
    size_t n = 0;
    TmpBuf() = default;
    explicit TmpBuf(size_t count) { alloc(count); }
    TmpBuf(const TmpBuf&) = delete;
    TmpBuf& operator=(const TmpBuf&) = delete;
    TmpBuf(TmpBuf&& o) noexcept : p(o.p), n(o.n) { o.p = nullptr; o.n = 0; }
    TmpBuf& operator=(TmpBuf&& o) noexcept {
        if (this != &o) { release(); p = o.p; n = o.n; o.p = nullptr; o.n = 0; }
        return *this;
    }
    ~TmpBuf() { release(); }
    void alloc(size_t count) {
        release();
        if (!count) return;
        p = static_cast<T*>(tl_arena->take(count * sizeof(T)));
        n = count;
    }
    void release() {
        if (p) tl_arena->give(p, n * sizeof(T));
        p = nullptr;
        n = 0;
    }
};

}  // namespace vcsrmc
