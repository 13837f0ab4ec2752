// srf_pool.hip -- device memory of plans and of one-shot scratch (srf_internal.hpp,
// pool_get / pool_put), and srf_plan_pool_trim.
//
// Blocks are hipMalloc'd in rounded sizes and kept when they are given back: at
// most POOL_KEEP bytes per device, and SCRATCH_KEEP of them from the scratch of calls
// that keep no plan, the oldest ones going to the system first.
// A block given back on a stream carries an event recorded there; whoever takes
// it next, on any stream or host thread, first lets its stream wait for that
// event.  The stream-ordered pool of the HIP runtime served this before: it
// returned the memory of several blocks freed in a row to the system, at about
// 0.25 ms per free and 0.05 ms per allocation (a plan frees 11 scratch buffers).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <list>
#include <mutex>
#include <unordered_map>

#include "srf_hip.h"
#include "srf_internal.hpp"

namespace {

constexpr uint64_t POOL_KEEP = 16ull << 30;
constexpr uint64_t SCRATCH_KEEP = 6ull << 30;   // one long backprojection takes up to about 4 GB
constexpr int POOL_DEVICES = 64;

struct Block {
    void *p;
    size_t bytes;
    int dev;
    hipEvent_t ev;     // recorded when the block was given back
    bool wait;         // the next user waits for ev
    bool scratch;      // given back by a call that keeps no plan
};

std::mutex mu;
std::unordered_map<void *, Block> &live()   // blocks in use (never destroyed: plans may outlive statics)
{
    static auto *m = new std::unordered_map<void *, Block>();
    return *m;
}
std::list<Block> &kept(int dev)             // blocks given back, oldest first
{
    static auto *l = new std::list<Block>[POOL_DEVICES];
    return l[dev];
}
uint64_t kept_bytes[POOL_DEVICES], kept_scratch[POOL_DEVICES];

int current_device()
{
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= POOL_DEVICES) {
        (void)hipGetLastError();
        return -1;
    }
    return dev;
}

// Sizes in steps of an eighth of their power of two (and of 64 KiB), so that
// blocks of nearly equal lists (the subsets of one scan) fit each other.
size_t rounded(size_t b)
{
    size_t step = 65536;
    while (step * 16 < b) step *= 2;
    return (b + step - 1) / step * step;
}

void release(Block &b)
{
    // hipFree waits for the device's work, so nothing still uses the block
    (void)hipFree(b.p);
    if (b.ev) (void)hipEventDestroy(b.ev);
}

// Takes a kept block out of its list.
Block take(std::list<Block>::iterator it, int dev)
{
    const Block b = *it;
    kept(dev).erase(it);
    kept_bytes[dev] -= b.bytes;
    if (b.scratch) kept_scratch[dev] -= b.bytes;
    return b;
}

// Releases kept blocks of the device, oldest first, down to keep bytes and scratch bytes.
void trim_locked(int dev, uint64_t keep, uint64_t scratch)
{
    auto &l = kept(dev);
    for (auto it = l.begin(); it != l.end() && (kept_bytes[dev] > keep || kept_scratch[dev] > scratch);) {
        const auto here = it++;
        if (kept_bytes[dev] <= keep && !here->scratch) continue;
        Block b = take(here, dev);
        release(b);
    }
}

// A new block of `want` bytes, or of `least` where the card has no more.
void *allocate(size_t want, size_t least, int dev, size_t &got)
{
    void *p = nullptr;
    for (int tries = 0; tries < 3; ++tries) {
        got = tries < 2 ? want : least;
        if (hipMalloc(&p, got) == hipSuccess) return p;
        (void)hipGetLastError();
        if (tries == 0) trim_locked(dev, 0, 0);
    }
    return nullptr;
}

}  // namespace

namespace srf {

void *pool_get(size_t bytes, hipStream_t s)
{
    const int dev = current_device();
    if (dev < 0) return nullptr;
    const size_t want = rounded(bytes ? bytes : 1);
    std::lock_guard<std::mutex> lock(mu);
    Block b{nullptr, 0, dev, nullptr, false, false};
    try {
        auto &l = kept(dev);
        // the smallest kept block that fits without wasting more than a quarter;
        // among equals the one given back last
        auto best = l.end();
        for (auto it = l.begin(); it != l.end(); ++it)
            if (it->bytes >= want && it->bytes - want <= want / 4 && (best == l.end() || it->bytes <= best->bytes)) best = it;
        if (best != l.end()) {
            if (best->wait && hipStreamWaitEvent(s, best->ev, 0) != hipSuccess) {
                (void)hipGetLastError();
                return nullptr;
            }
            b = take(best, dev);
        } else {
            b.p = allocate(want, bytes ? bytes : 1, dev, b.bytes);
            if (!b.p) return nullptr;
        }
        live()[b.p] = b;
        return b.p;
    } catch (...) {   // no host memory for the pool's own lists
        if (b.p) release(b);
        return nullptr;
    }
}

void pool_put(void *p, hipStream_t s, bool idle, bool scratch)
{
    if (!p) return;
    std::lock_guard<std::mutex> lock(mu);
    auto it = live().find(p);
    if (it == live().end()) return;
    Block b = it->second;
    live().erase(it);
    b.wait = false;
    b.scratch = scratch;
    if (!idle) {
        if ((b.ev || hipEventCreateWithFlags(&b.ev, hipEventDisableTiming) == hipSuccess) &&
            hipEventRecord(b.ev, s) == hipSuccess) {
            b.wait = true;
        } else {
            (void)hipGetLastError();
            release(b);   // no event to order a later use by
            return;
        }
    }
    try {
        kept(b.dev).push_back(b);
    } catch (...) {
        release(b);
        return;
    }
    kept_bytes[b.dev] += b.bytes;
    if (scratch) kept_scratch[b.dev] += b.bytes;
    trim_locked(b.dev, POOL_KEEP, SCRATCH_KEEP);
}

}  // namespace srf

extern "C" int srf_plan_pool_trim(size_t keep_bytes)
{
    const int dev = current_device();
    if (dev < 0) return SRF_ERR_LAUNCH;
    if (hipDeviceSynchronize() != hipSuccess) {
        (void)hipGetLastError();
        return SRF_ERR_LAUNCH;
    }
    std::lock_guard<std::mutex> lock(mu);
    trim_locked(dev, keep_bytes, keep_bytes);
    return SRF_OK;
}
