"""The device block pool (srf_pool.hip) on the host, compiled against a small model of the
HIP calls it makes: streams with vector clocks, events, a card of limited memory.

The model counts a violation when a block is used on a stream that is not ordered after the
block's last use on another one, when a block is handed to two users, and when memory that
is not allocated is freed or waited for work is."""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#pragma once
#include <stddef.h>
#include <stdint.h>
typedef void *hipStream_t;
typedef void *hipEvent_t;
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone = 0 };
constexpr unsigned hipEventDisableTiming = 2;
hipError_t hipMalloc(void **p, size_t n);
hipError_t hipFree(void *p);
hipError_t hipGetDevice(int *d);
hipError_t hipGetLastError();
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned);
hipError_t hipEventDestroy(hipEvent_t e);
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s);
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned);
hipError_t hipDeviceSynchronize();
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st);
"""

MODEL = r"""
#include <map>
#include <mutex>
#include <new>
#include <random>
#include <stdlib.h>
#include <thread>
#include <vector>
#include "hip/hip_runtime.h"

constexpr int NS = 8;   // streams 1..NS, as handles
struct Clock { long t[NS + 1] = {}; };
struct Use { int stream = 0; long t = 0; size_t bytes = 0; bool owned = false; };
std::mutex sim;
Clock stream[NS + 1];
std::map<void *, Use> mem;
std::map<void *, Clock> event;
size_t limit = ~(size_t)0, used = 0, peak = 0;
uintptr_t next_p = 1 << 20;
long violations = 0, mallocs = 0, frees = 0;
bool fail_record = false, fail_wait = false;
thread_local long throw_after = -1;   // operator new fails after this many calls

void *operator new(size_t n)
{
    if (throw_after >= 0 && throw_after-- == 0) throw std::bad_alloc();
    void *p = malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

struct NoThrow {   // the model's own containers never fail
    long keep = throw_after;
    NoThrow() { throw_after = -1; }
    ~NoThrow() { throw_after = keep; }
};

hipError_t hipMalloc(void **p, size_t n)
{
    NoThrow q;
    std::lock_guard<std::mutex> l(sim);
    if (used + n > limit) return hipErrorOutOfMemory;
    *p = (void *)next_p;
    next_p += n + 4096;
    used += n;
    peak = used > peak ? used : peak;
    mem[*p].bytes = n;
    ++mallocs;
    return hipSuccess;
}
hipError_t hipFree(void *p)   // waits for the device
{
    NoThrow q;
    std::lock_guard<std::mutex> l(sim);
    auto it = mem.find(p);
    if (it == mem.end() || it->second.owned) { ++violations; return hipErrorUnknown; }
    used -= it->second.bytes;
    mem.erase(it);
    ++frees;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    NoThrow q;
    std::lock_guard<std::mutex> l(sim);
    *e = (void *)(next_p += 4096);
    event[*e];
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    NoThrow q;
    std::lock_guard<std::mutex> l(sim);
    if (!event.erase(e)) ++violations;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    NoThrow q;
    std::lock_guard<std::mutex> l(sim);
    if (fail_record) return hipErrorUnknown;
    if (!event.count(e)) ++violations;
    event[e] = stream[(intptr_t)s];
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    NoThrow q;
    std::lock_guard<std::mutex> l(sim);
    if (fail_wait) return hipErrorUnknown;
    if (!event.count(e)) { ++violations; return hipErrorUnknown; }
    for (int k = 0; k <= NS; ++k)
        if (event[e].t[k] > stream[(intptr_t)s].t[k]) stream[(intptr_t)s].t[k] = event[e].t[k];
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *st) { *st = hipStreamCaptureStatusNone; return hipSuccess; }

#include "srf_internal.hpp"

// Kernels on the block, queued on stream s.
static void use(void *p, int s, size_t bytes)
{
    NoThrow q;
    std::lock_guard<std::mutex> l(sim);
    auto it = mem.find(p);
    if (it == mem.end() || it->second.bytes < bytes) { ++violations; return; }
    Use &u = it->second;
    if (u.stream && u.stream != s && stream[s].t[u.stream] < u.t) ++violations;   // not ordered after the last use
    u.stream = s;
    u.t = ++stream[s].t[s];
}
static void own(void *p, bool on)
{
    NoThrow q;
    std::lock_guard<std::mutex> l(sim);
    auto it = mem.find(p);
    if (it == mem.end() || it->second.owned == on) { ++violations; return; }
    it->second.owned = on;
}
static void synchronize(int s)   // the host waits for s: every stream's later work follows it
{
    std::lock_guard<std::mutex> l(sim);
    for (int k = 1; k <= NS; ++k)
        for (int j = 0; j <= NS; ++j)
            if (stream[s].t[j] > stream[k].t[j]) stream[k].t[j] = stream[s].t[j];
}

extern "C" {
int srf_plan_pool_trim(size_t);
void *get(size_t n, int s)
{
    void *p = srf::pool_get(n, (hipStream_t)(intptr_t)s);
    if (p) { own(p, true); use(p, s, n); }
    return p;
}
void put(void *p, int s, int idle, int scratch)
{
    if (idle) synchronize(s);
    own(p, false);
    srf::pool_put(p, (hipStream_t)(intptr_t)s, idle, scratch);
}
void use_block(void *p, int s) { use(p, s, 0); }
void raw_put(void *p) { srf::pool_put(p, nullptr, false, false); }
// Threads that take, use and give back blocks of a few sizes, each on a stream of its own
// or on shared ones.
long run_threads(int threads, int steps, int shared, int seed)
{
    std::vector<std::thread> ts;
    for (int i = 0; i < threads; ++i)
        ts.emplace_back([=] {
            std::mt19937 r(seed + i);
            std::vector<std::pair<void *, int>> held;
            for (int k = 0; k < steps; ++k) {
                const int s = shared ? 1 + (int)(r() % NS) : 1 + i % NS;
                if (held.size() < 6 && r() % 2) {
                    const size_t n = (size_t)(1 + r() % 5) << 20;
                    if (void *p = get(n, s)) held.emplace_back(p, s);
                } else if (!held.empty()) {
                    const size_t j = r() % held.size();
                    use_block(held[j].first, held[j].second);
                    put(held[j].first, held[j].second, r() % 4 == 0, r() % 2);
                    held.erase(held.begin() + (long)j);
                }
            }
            for (auto &h : held) put(h.first, h.second, 0, 0);
        });
    for (auto &t : ts) t.join();
    return violations;
}
void set_limit(size_t n) { limit = n; }
void set_fail(int record, int wait) { fail_record = record; fail_wait = wait; }
void set_throw(long after) { throw_after = after; }
long count_violations() { return violations; }
size_t in_use() { return used; }
size_t peak_use() { return peak; }
long count_mallocs() { return mallocs; }
}
"""


@pytest.fixture(scope="module")
def shared_object(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("pool")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "model.cpp").write_text(MODEL)
    shutil.copy(os.path.join(ROOT, "srf_amd", "csrc", "srf_pool.hip"), d / "pool.cpp")
    so = d / "libpool.so"
    subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-fPIC", "-shared", "-pthread", "-I", str(d),
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "srf_amd", "csrc"),
                    str(d / "model.cpp"), str(d / "pool.cpp"), "-o", str(so)], check=True)
    return so


@pytest.fixture
def pool(shared_object, tmp_path):
    """A pool of its own for every test (a copy of the library, loaded afresh)."""
    so = tmp_path / "libpool.so"
    shutil.copy(shared_object, so)
    L = ctypes.CDLL(str(so), mode=os.RTLD_LOCAL | os.RTLD_NOW)
    L.get.restype = ctypes.c_void_p
    L.get.argtypes = [ctypes.c_size_t, ctypes.c_int]
    L.put.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    L.use_block.argtypes = [ctypes.c_void_p, ctypes.c_int]
    L.set_limit.argtypes = [ctypes.c_size_t]
    L.set_throw.argtypes = [ctypes.c_long]
    L.srf_plan_pool_trim.argtypes = [ctypes.c_size_t]
    for f in (L.run_threads, L.count_violations, L.count_mallocs):
        f.restype = ctypes.c_long
    L.in_use.restype = L.peak_use.restype = ctypes.c_size_t
    yield L
    assert L.count_violations() == 0


def test_reuse_on_another_stream_is_ordered(pool):
    p = pool.get(1 << 20, 1)
    pool.put(p, 1, 0, 0)
    q = pool.get(1 << 20, 2)     # the model counts a violation if stream 2 did not wait
    assert q == p and pool.count_mallocs() == 1
    pool.put(q, 2, 1, 0)
    assert pool.get(1 << 20, 3) == p


@pytest.mark.parametrize("shared", [0, 1])
@pytest.mark.parametrize("threads", [2, 8])
def test_threads_and_streams(pool, threads, shared):
    assert pool.run_threads(threads, 4000, shared, 7 * threads + shared) == 0
    assert pool.srf_plan_pool_trim(0) == 0
    assert pool.in_use() == 0


def test_kept_memory_is_bounded_and_given_back(pool):
    G = 1 << 30
    blocks = [pool.get(G, 1) for _ in range(20)]
    for p in blocks:
        pool.put(p, 1, 0, 0)
    assert pool.in_use() == 16 * G
    assert pool.srf_plan_pool_trim(3 * G) == 0 and pool.in_use() == 3 * G
    assert pool.srf_plan_pool_trim(0) == 0 and pool.in_use() == 0


def test_scratch_is_kept_less(pool):
    G = 1 << 30
    plan = [pool.get(G, 1) for _ in range(4)]
    scratch = [pool.get(2 * G, 1) for _ in range(5)]
    for p in plan:
        pool.put(p, 1, 1, 0)
    for p in scratch:
        pool.put(p, 1, 0, 1)
    assert pool.in_use() == 4 * G + 6 * G    # the plans' blocks stay, three of the scratch ones
    # a scratch block that a plan takes and gives back counts as the plan's
    q = pool.get(2 * G, 1)
    pool.put(q, 1, 0, 0)
    more = [pool.get(3 * G, 1) for _ in range(3)]
    for p in more:
        pool.put(p, 1, 0, 1)
    assert pool.in_use() == 4 * G + 2 * G + 6 * G


def test_the_last_memory_of_the_card(pool):
    """A block whose rounded size does not fit any more, but whose size does."""
    M = 1 << 20
    n = 100 * M + 1000
    pool.set_limit(n)
    keep = pool.get(2 * M, 1)
    pool.put(keep, 1, 0, 0)                  # kept memory goes to the system first
    p = pool.get(n, 1)
    assert p and pool.in_use() == n
    assert not pool.get(M, 1)
    pool.put(p, 1, 0, 0)


def test_failing_calls(pool):
    p = pool.get(1 << 20, 1)
    pool.set_fail(1, 0)
    pool.put(p, 1, 0, 0)                     # no event to order a later use by: freed
    assert pool.in_use() == 0
    pool.set_fail(0, 0)
    q = pool.get(1 << 20, 1)
    pool.put(q, 1, 0, 0)
    pool.set_fail(0, 1)
    assert not pool.get(1 << 20, 2)          # cannot wait: none, and the block stays kept
    pool.set_fail(0, 0)
    assert pool.get(1 << 20, 2) == q


def test_no_host_memory(pool):
    """operator new failing inside the pool: null or a freed block, no exception."""
    for after in range(6):
        before = pool.in_use()
        pool.set_throw(after)
        p = pool.get((3 + after) << 20, 1)
        pool.set_throw(-1)
        if not p:
            assert pool.in_use() == before
            continue
        for late in range(4):
            pool.set_throw(late)
            pool.put(p, 1, 0, 0)
            pool.set_throw(-1)
            p = pool.get((3 + after) << 20, 1)
            assert p
        pool.put(p, 1, 1, 0)
    pool.srf_plan_pool_trim(0)
    assert pool.in_use() == 0
