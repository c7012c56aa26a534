// Device memory of the library's buffers: a bounded cache of freed allocations in front
// of hipMalloc / hipFree.
//
// A build allocates about 20 arrays and a device-pointer query about 8; straight from the
// runtime that cost more than the kernels (2M-triangle LBVH build and collapse with the
// previous tree destroyed: 5.0 ms a pass against 0.7 ms of kernels; a batch of 64 scenes
// built and queried: 9.0 against 1.0), since every hipMalloc maps and every hipFree drains
// the device and unmaps.
//
// Rules:
//   * a block enters the cache only when the device has no work left that could touch it:
//     devFree waits for the device first, as hipFree does, unless the caller has just
//     waited itself (QuietFree).  A cached block may therefore be handed to any thread and
//     used on any stream at once;
//   * blocks are kept per device and handed out again on that device only;
//   * at most kMaxCached bytes per device stay cached (the longest unused go first).  Every
//     allocation and every free gives back the blocks that have lain for longer than
//     kMaxIdle (there is no thread that does: a program that only queries resident buffers,
//     or stops, keeps them until then); an allocation that fails gives all of them back
//     before it tries again; qr_dev_trim gives them back on request;
//   * sizes are rounded up to multiples of 512 bytes and, from 4 KiB on, by at most an
//     eighth; a request takes a cached block of up to one and a half times its size;
//   * nothing is kept for a pointer the cache did not hand out: devFree passes it on.
#include <chrono>
#include <list>
#include <map>
#include <mutex>
#include <new>
#include <unordered_map>

#include "qr_internal.h"

namespace qr {

namespace {

constexpr size_t kMaxCached = size_t(4) << 30;
constexpr auto kMaxIdle = std::chrono::seconds(10);

using Clock = std::chrono::steady_clock;

struct Block {
    size_t size = 0;
    int dev = 0;
    bool cached = false;
    Clock::time_point since{};                      // cached: when it was freed
    std::list<void*>::iterator age{};               //   its place in the device's lists
    std::multimap<size_t, void*>::iterator bySize{};
};

struct Cached {
    std::list<void*> byAge;  // longest unused first
    std::multimap<size_t, void*> bySize;
    size_t bytes = 0;
};

struct Pool {
    std::mutex m;
    std::unordered_map<void*, Block> blocks;  // handed out or cached
    std::map<int, Cached> cached;             // by device
};

// never destroyed: buffers may be released by other static destructors
Pool& pool() {
    static Pool* p = new Pool;
    return *p;
}

size_t roundUp(size_t bytes) {
    size_t step = 512;
    while (step * 16 <= bytes) step <<= 1;
    return (bytes + step - 1) / step * step;
}

// (the lock is held by the callers of these)
void uncache(Cached& c, Block& b) {
    c.byAge.erase(b.age);
    c.bySize.erase(b.bySize);
    c.bytes -= b.size;
    b.cached = false;
}

// Cached blocks to give back now, taken off the books: all of the device's, or those idle
// for too long and, while more than kMaxCached are cached, the longest unused.  (Without
// memory for the list the rest stays cached.)
std::vector<void*> excess(Pool& P, int dev, bool all) {
    std::vector<void*> out;
    Cached& c = P.cached[dev];
    const auto now = Clock::now();
    try {
        while (!c.byAge.empty()) {
            void* p = c.byAge.front();
            const auto it = P.blocks.find(p);
            if (!all && c.bytes <= kMaxCached && now - it->second.since <= kMaxIdle) break;
            out.push_back(p);
            uncache(c, it->second);
            P.blocks.erase(it);
        }
    } catch (const std::bad_alloc&) {
    }
    return out;
}

void giveBack(const std::vector<void*>& blocks) {
    for (void* p : blocks) (void)hipFree(p);
}

thread_local int tQuiet = 0;

}  // namespace

void QuietFree::begin() {
    if (!on) ++tQuiet;
    on = true;
}
QuietFree::~QuietFree() {
    if (on) --tQuiet;
}

void* devAlloc(size_t bytes) {
    int dev = 0;
    hipCheck(hipGetDevice(&dev), "get device");
    const size_t want = roundUp(bytes > 0 ? bytes : 1);
    Pool& P = pool();
    void* p = nullptr;
    std::vector<void*> back;
    {
        std::lock_guard<std::mutex> lock(P.m);
        Cached& c = P.cached[dev];
        const auto it = c.bySize.lower_bound(want);
        if (it != c.bySize.end() && it->first <= want + want / 2) {
            p = it->second;
            uncache(c, P.blocks[p]);
        }
        back = excess(P, dev, false);
    }
    giveBack(back);
    if (p) return p;
    hipError_t e = hipMalloc(&p, want);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        devTrim();
        e = hipMalloc(&p, want);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        throw OomError(std::string("hipMalloc failed: ") + hipGetErrorString(e));
    }
    std::lock_guard<std::mutex> lock(P.m);
    Block b;
    b.size = want;
    b.dev = dev;
    P.blocks[p] = b;
    return p;
}

hipError_t devFree(void* p) {
    if (!p) return hipSuccess;
    int dev = 0;
    Pool& P = pool();
    bool known = false, mine = false;
    {
        std::lock_guard<std::mutex> lock(P.m);
        const auto it = P.blocks.find(p);
        known = it != P.blocks.end();
        if (known && it->second.cached) return hipErrorInvalidValue;  // freed already
        mine = known && hipGetDevice(&dev) == hipSuccess && it->second.dev == dev;
        if (known && !mine) P.blocks.erase(it);
    }
    // not the cache's, or of another device than the current one: the runtime's own free
    if (!mine) return hipFree(p);
    if (tQuiet == 0) {
        const hipError_t e = hipDeviceSynchronize();
        if (e != hipSuccess) {  // the device has failed: keep nothing
            {
                std::lock_guard<std::mutex> lock(P.m);
                P.blocks.erase(p);
            }
            (void)hipFree(p);
            return e;
        }
    }
    std::vector<void*> back;
    try {
        std::lock_guard<std::mutex> lock(P.m);
        Cached& c = P.cached[dev];
        Block& b = P.blocks.at(p);
        if (b.cached) return hipErrorInvalidValue;
        const auto bySize = c.bySize.emplace(b.size, p);
        try {
            b.age = c.byAge.insert(c.byAge.end(), p);
        } catch (...) {
            c.bySize.erase(bySize);
            throw;
        }
        b.bySize = bySize;
        b.cached = true;
        b.since = Clock::now();
        c.bytes += b.size;
        p = nullptr;  // cached
        back = excess(P, dev, false);
    } catch (...) {  // no memory for the books: buffers are released by destructors, which must not throw
        if (p) {
            std::lock_guard<std::mutex> lock(P.m);
            P.blocks.erase(p);
        }
        if (p) (void)hipFree(p);
    }
    giveBack(back);
    return hipSuccess;
}

void devTrim() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return;
    Pool& P = pool();
    std::vector<void*> back;
    {
        std::lock_guard<std::mutex> lock(P.m);
        back = excess(P, dev, true);
    }
    giveBack(back);
}

int* pinnedInts() {
    static thread_local int* w = nullptr;
    if (!w) hipCheck(hipHostMalloc(reinterpret_cast<void**>(&w), 16 * sizeof(int), hipHostMallocDefault), "pinned words");
    return w;
}

int* pinnedIntsDevice() {
    static thread_local int* d = nullptr;
    if (!d) hipCheck(hipHostGetDevicePointer(reinterpret_cast<void**>(&d), pinnedInts(), 0), "pinned words map");
    return d;
}

}  // namespace qr
