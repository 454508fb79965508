// The library's device memory (vcsr_mc_amd/csrc/device_memory.hpp) on a stand-in for the runtime: a
// card of a given size whose allocations are numbers.  Prints "ok", or the check that failed.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <random>
#include <thread>

#include "../../vcsr_mc_amd/csrc/device_memory.hpp"

namespace card {
std::mutex m;
size_t size = 0, used = 0;
uintptr_t next = 4096;
std::map<uintptr_t, size_t> live;
thread_local int device = 0;
}  // namespace card

#define CHECK(cond)                                                          \
    do {                                                                     \
        if (!(cond)) {                                                       \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #cond);           \
            std::exit(1);                                                    \
        }                                                                    \
    } while (0)

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
    std::lock_guard<std::mutex> lock(card::m);
    if (card::used + bytes > card::size) return hipErrorOutOfMemory;
    card::used += bytes;
    card::live[card::next] = bytes;
    *p = reinterpret_cast<void*>(card::next);
    card::next += (bytes + 4095) / 4096 * 4096 + 4096;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (!p) return hipSuccess;
    std::lock_guard<std::mutex> lock(card::m);
    const auto it = card::live.find(reinterpret_cast<uintptr_t>(p));
    CHECK(it != card::live.end());  // freed twice, or never allocated
    card::used -= it->second;
    card::live.erase(it);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* free_bytes, size_t* total) {
    std::lock_guard<std::mutex> lock(card::m);
    *free_bytes = card::size - card::used;
    *total = card::size;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipGetDevice(int* d) {
    *d = card::device;
    return hipSuccess;
}
}

namespace vcsrmc {
[[noreturn]] void throw_hip(hipError_t e, const char* what, const char*, int) {
    throw Error((int)e, what);
}
}  // namespace vcsrmc

using namespace vcsrmc;

static constexpr size_t MB = (size_t)1 << 20, GB = (size_t)1 << 30;

static void start(size_t bytes) {
    BlockCache::instance().give_back_all();
    CHECK(card::used == 0);
    card::size = bytes;
}

// A call that takes `bytes` of scratch at once and waits for its stream.
static void call(size_t bytes) {
    ScratchScope scratch(bytes);
    TmpBuf<char> t(bytes);
    scratch.idle();
}

template <typename Fn>
static bool out_of_memory(Fn&& fn) {
    try {
        fn();
    } catch (const Error& e) {
        CHECK(e.status == (int)hipErrorOutOfMemory);
        return true;
    }
    return false;
}

// An allocation fails only for want of memory that the library itself does not hold idle.
static void kept_blocks_are_given_back() {
    start(3 * GB);
    call(GB);
    CHECK(card::used >= GB);  // kept
    {
        DevBuf<char> format(2 * GB + 512 * MB);  // a format's array, a binary16 copy of B
        CHECK(card::used == 2 * GB + 512 * MB);
    }
    call(GB);
    {
        ScratchScope scratch(2 * GB + 512 * MB);  // another call's scratch
        TmpBuf<char> t(2 * GB + 512 * MB);
    }
    call(GB);
    void* p = nullptr;
    CHECK(device_malloc(&p, 2 * GB + 512 * MB) == hipSuccess);
    CHECK(hipFree(p) == hipSuccess);
    call(GB);
    CHECK(out_of_memory([] { DevBuf<char> b(3 * GB + 1); }));
    CHECK(card::used == 0);
}

// ... nor in this call's own blocks that nothing uses at the time.
static void unused_blocks_of_the_call_are_given_back() {
    start(3 * GB);
    ScratchScope scratch(0);
    TmpBuf<char> small(64);
    {
        TmpBuf<char> large(2 * GB);
    }
    DevBuf<char> format(2 * GB);
    TmpBuf<char> again(512 * MB);
    CHECK(out_of_memory([] { TmpBuf<char> t(GB); }));
}

// What a call can use does not depend on what it has reserved or what earlier calls left.
static void available_counts_idle_memory() {
    start(64 * GB);
    call(GB);
    ScratchScope scratch(2 * GB);
    CHECK(tl_arena->available() == 64 * GB);
    TmpBuf<char> a(512 * MB);
    CHECK(tl_arena->available() == 64 * GB - 512 * MB);
    DevBuf<char> format(GB);
    {
        TmpBuf<char> b(8 * GB);
        CHECK(tl_arena->available() == 64 * GB - 512 * MB - 9 * GB);
    }
    CHECK(tl_arena->available() == 64 * GB - 512 * MB - GB);
}

// Scratch is reserved ahead only where there is room for what lasts; else it grows as asked for.
static void large_reserves_need_room() {
    start(64 * GB);
    {
        ScratchScope scratch(12 * GB);
        TmpBuf<char> a(MB);
        CHECK(card::used == 12 * GB);
    }
    CHECK(card::used == 0);
    {
        DevBuf<char> others(40 * GB);
        ScratchScope scratch(12 * GB);
        TmpBuf<char> a(MB), b(GB);
        CHECK(card::used < 42 * GB);
        DevBuf<char> format(22 * GB);
    }
    CHECK(card::used == 0);
}

// A block stays for 16 calls that do not take it, however many blocks those use.
static void blocks_age_by_calls() {
    start(64 * GB);
    call(100 * MB);
    const uintptr_t block = card::live.begin()->first;
    for (int i = 0; i < 17; ++i) {
        CHECK(card::live.count(block) == 1);
        ScratchScope scratch(200 * MB);
        TmpBuf<char> a(200 * MB), b(220 * MB), c(240 * MB);
        scratch.idle();
    }
    CHECK(card::live.count(block) == 0);
}

// At most 2 GiB are kept, the youngest; a call that asks for a word takes and leaves a word.
static void kept_memory_is_bounded() {
    start(64 * GB);
    for (size_t size = 100 * MB; size < 3 * GB; size += 300 * MB) {
        call(size);
        CHECK(card::used <= 2 * GB);
    }
    start(64 * GB);
    {
        ScratchScope scratch(0);
        TmpBuf<unsigned> word(1);
        CHECK(card::used <= 4096);
        scratch.idle();
    }
    CHECK(card::used <= 4096);
}

// Ranges in use at the same time never overlap, lie in live blocks, and all goes back.
static void ranges_are_apart() {
    start(64 * GB);
    std::mt19937_64 rng(1);
    for (int round = 0; round < 50; ++round) {
        ScratchScope scratch(rng() % (256 * MB));
        std::vector<TmpBuf<char>> held;
        for (int i = 0; i < 200; ++i) {
            if (!held.empty() && rng() % 2) {
                std::swap(held[rng() % held.size()], held.back());
                held.pop_back();
                continue;
            }
            held.emplace_back(1 + rng() % ((size_t)1 << (rng() % 27)));
            std::map<uintptr_t, size_t> at;
            for (const auto& t : held) at[reinterpret_cast<uintptr_t>(t.p)] = t.n;
            CHECK(at.size() == held.size());
            uintptr_t end = 0;
            for (const auto& [p, n] : at) {
                CHECK(p >= end);
                end = p + n;
                const auto block = --card::live.upper_bound(p);
                CHECK(end <= block->first + block->second);
            }
        }
        held.clear();
        if (round % 3) scratch.idle();
    }
    BlockCache::instance().give_back_all();
    CHECK(card::used == 0);
}

// A call that ends in an error keeps nothing: its kernels may still run.
static void failed_calls_keep_nothing() {
    start(4 * GB);
    try {
        ScratchScope scratch(GB);
        TmpBuf<char> t(GB);
        throw Error(1, "refused");
    } catch (const Error&) {
    }
    CHECK(card::used == 0);
}

static void threads() {
    start(200 * GB);
    std::vector<std::thread> all;
    for (int t = 0; t < 8; ++t)
        all.emplace_back([t] {
            card::device = t % 2;
            std::mt19937_64 rng(t);
            for (int i = 0; i < 300; ++i) {
                call(1 + rng() % (300 * MB));
                if (rng() % 16 == 0) BlockCache::instance().give_back_all();
            }
        });
    for (auto& t : all) t.join();
    CHECK(card::used <= 2 * GB);
    BlockCache::instance().give_back_all();
    CHECK(card::used == 0);
}

int main(int argc, char** argv) {
    const std::pair<const char*, void (*)()> checks[] = {
        {"kept_blocks_are_given_back", kept_blocks_are_given_back},
        {"unused_blocks_of_the_call_are_given_back", unused_blocks_of_the_call_are_given_back},
        {"available_counts_idle_memory", available_counts_idle_memory},
        {"large_reserves_need_room", large_reserves_need_room},
        {"blocks_age_by_calls", blocks_age_by_calls},
        {"kept_memory_is_bounded", kept_memory_is_bounded},
        {"ranges_are_apart", ranges_are_apart},
        {"failed_calls_keep_nothing", failed_calls_keep_nothing},
        {"threads", threads},
    };
    for (const auto& [name, check] : checks)
        if (argc == 2 && std::strcmp(argv[1], name) == 0) {
            check();
            std::puts("ok");
            return 0;
        }
    std::puts("no such check");
    return 1;
}
