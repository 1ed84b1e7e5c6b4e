// handoff.hip -- staged copies between caller host memory and HBM: walk
// buffers out to caller-owned host arrays, edge batches in.
//
// The reference fills its host walk set with one blocking cudaMemcpy per array
// into malloc'd memory (data/walk_set/walk_set_host.cu:55-85).  On this host a
// plain D2H copy into fresh pageable memory runs at a few GB/s: the runtime
// stages through its own small pinned buffer on one thread, and every 4 KiB
// page of the destination faults on first touch.  Here:
//  - destinations are 2 MiB-aligned and advised for transparent huge pages,
//    so first touch faults once per 2 MiB (they stay malloc-compatible:
//    free() releases them, as the C ABI promises);
//  - the copy is split into chunks that several host threads pull from one
//    queue; each thread owns a lane -- a HIP stream and two pinned staging
//    buffers -- so the DMA of its next chunk overlaps its memcpy of the current
//    one, and the page faults of the destination are taken by all threads at
//    once; chunks shrink with the copy, so that a few MB still spread;
//  - a copy of at most kPackBelow goes through one pinned buffer with one
//    kernel on the engine's stream that moves every array (a runtime copy of
//    pageable memory costs some 10 us per array): walks from 32 seeds 156 ->
//    120 us.
// Lanes are kept in a pool per device, shared by its handles, until the last of
// them ends: pinning their 16 MiB takes longer than most copies, and a handle
// beside others need not pay it again.
// Host-pointer ingest (trw_add_edges) uses the same lanes in the other
// direction: the reference copies each batch array with one blocking
// cudaMemcpy (data/buffer.cuh:135-149).
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <thread>

#include "engine.h"

namespace trw {

namespace {

constexpr size_t kHuge = size_t(2) << 20;
constexpr size_t kChunk = kStageBytes;            // bytes of a staging buffer
constexpr size_t kMinChunk = size_t(512) << 10;   // smallest staged chunk
constexpr size_t kPackBelow = size_t(2) << 20;    // smaller copies: one kernel
constexpr int kMaxThreads = 32;

int copy_threads() {
    static const int n = [] {
        int t = 8;
        if (const char* s = getenv("TRW_HOST_COPY_THREADS")) t = atoi(s);
        return std::max(1, std::min(t, kMaxThreads));
    }();
    return n;
}

// The lanes not in use, per device.  At most kMaxThreads are kept on a device;
// its last engine's end frees them.  (The pool itself is never destroyed:
// nothing may call the runtime as the process ends.)
struct LanePool {
    struct Device {
        std::vector<std::unique_ptr<HostLane>> free;
        int engines = 0;
    };
    std::mutex mu;
    std::map<int, Device> devices;
};
LanePool& lane_pool() {
    static LanePool* pool = new LanePool;
    return *pool;
}

// Lanes of the current device taken from the pool for one copy.
struct Lanes {
    int device;
    std::vector<std::unique_ptr<HostLane>> v;
    Lanes(int dev, int n) : device(dev), v(take_lanes(dev, n)) {}
    ~Lanes() { give_lanes(device, v); }
};

// Up to kMaxSegs spans copied by one kernel, 16 bytes per thread: span i is the
// units [at[i], at[i + 1]).  Every span starts 16-byte aligned on both sides.
constexpr int kMaxSegs = 6;
struct PackArgs {
    const char* src[kMaxSegs];
    char* dst[kMaxSegs];
    uint64_t bytes[kMaxSegs];
    uint64_t at[kMaxSegs + 1];
    int n;
};
__global__ __launch_bounds__(256) void pack_kernel(PackArgs a) {
    const uint64_t i = blockIdx.x * 256ull + threadIdx.x;
    if (i >= a.at[a.n]) return;
    int k = 0;
    while (i >= a.at[k + 1]) ++k;
    const uint64_t o = (i - a.at[k]) * 16;
    if (o + 16 <= a.bytes[k]) {
        *reinterpret_cast<uint4*>(a.dst[k] + o) = *reinterpret_cast<const uint4*>(a.src[k] + o);
    } else {
        for (uint64_t b = o; b < a.bytes[k]; ++b) a.dst[k][b] = a.src[k][b];
    }
}

}  // namespace

std::vector<std::unique_ptr<HostLane>> take_lanes(int device, int n) {
    if (alloc_hook_fires(g_alloc_fail_after)) throw std::bad_alloc();
    std::vector<std::unique_ptr<HostLane>> v;
    {
        LanePool& p = lane_pool();
        std::lock_guard<std::mutex> g(p.mu);
        auto& f = p.devices[device].free;
        while (static_cast<int>(v.size()) < n && !f.empty()) {
            v.push_back(std::move(f.back()));
            f.pop_back();
        }
    }
    while (static_cast<int>(v.size()) < n) v.push_back(std::make_unique<HostLane>());
    return v;
}

void give_lanes(int device, std::vector<std::unique_ptr<HostLane>>& lanes) {
    std::vector<std::unique_ptr<HostLane>> rest;  // freed outside the lock
    LanePool& p = lane_pool();
    std::lock_guard<std::mutex> g(p.mu);
    auto& d = p.devices[device];
    for (auto& l : lanes) {
        if (d.engines > 0 && d.free.size() < kMaxThreads) d.free.push_back(std::move(l));
        else rest.push_back(std::move(l));
    }
    lanes.clear();
}

char* StageLease::take() {
    lane = take_lanes(device, 1);
    lane[0]->init();
    return static_cast<char*>(lane[0]->stage[0]);
}

void StageLease::done() {
    if (!lane.empty()) give_lanes(device, lane);
}

StageLease::~StageLease() {
    if (lane.empty()) return;
    (void)hipStreamSynchronize(s);
    give_lanes(device, lane);
}

void attach_lanes(int device) {
    std::lock_guard<std::mutex> g(lane_pool().mu);
    ++lane_pool().devices[device].engines;
}

void detach_lanes(int device) {
    std::vector<std::unique_ptr<HostLane>> done;
    std::lock_guard<std::mutex> g(lane_pool().mu);
    auto& d = lane_pool().devices[device];
    if (--d.engines == 0) done.swap(d.free);
}

void* host_output_alloc(size_t bytes) {
    if (bytes < kHuge) {
        void* p = malloc(bytes ? bytes : 1);
        if (!p) throw std::bad_alloc();
        return p;
    }
    void* p = nullptr;
    if (posix_memalign(&p, kHuge, bytes) != 0 || !p) throw std::bad_alloc();
    // advisory only: without THP support the memory is simply 4 KiB-paged
    (void)madvise(p, (bytes + 4095) & ~size_t(4095), MADV_HUGEPAGE);
    return p;
}

HostLane::~HostLane() {
    if (stream) (void)hipStreamSynchronize(stream);
    for (auto& e : done)
        if (e) (void)hipEventDestroy(e);
    for (auto& b : stage)
        if (b) (void)hipHostFree(b);
    if (stream) (void)hipStreamDestroy(stream);
}

void HostLane::init() {
    if (!stream)
        check_hip(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking), "hipStreamCreate");
    for (auto& b : stage)
        if (!b) check_hip(hipHostMalloc(&b, kChunk, hipHostMallocDefault), "hipHostMalloc");
    for (auto& e : done)
        if (!e) check_hip(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
}

void Engine::copy_staged(const HostCopy* segs, size_t nseg, bool to_device) {
    copy_on_lanes(segs, nseg, to_device, true);
}

std::string Engine::join_prefetch() {
    if (!pf_pending) return "";
    if (pf_thread.joinable()) pf_thread.join();
    pf_pending = false;
    std::string err;
    err.swap(pf_error);
    return err;
}

void Engine::copy_on_lanes(const HostCopy* segs, size_t nseg, bool to_device, bool engine_order) {
    size_t total = 0, units = 0;
    for (size_t i = 0; i < nseg; ++i) {
        total += segs[i].bytes;
        units += (segs[i].bytes + 15) / 16;
    }
    // earlier work on the engine stream may still read or write these buffers
    if (engine_order) sync();
    const auto t0 = std::chrono::steady_clock::now();

    if (total == 0) {
        // nothing to copy
    } else if (units * 16 <= kPackBelow && nseg <= kMaxSegs) {
        Lanes ls(device, 1);
        ls.v[0]->init();
        hipStream_t st = engine_order ? stream : ls.v[0]->stream;
        char* stage = static_cast<char*>(ls.v[0]->stage[0]);
        PackArgs a{};
        for (size_t i = 0; i < nseg; ++i) {
            if (!segs[i].bytes) continue;
            char* at = stage + a.at[a.n] * 16;
            if (to_device) memcpy(at, segs[i].src, segs[i].bytes);
            a.src[a.n] = to_device ? at : static_cast<const char*>(segs[i].src);
            a.dst[a.n] = to_device ? static_cast<char*>(segs[i].dst) : at;
            a.bytes[a.n] = segs[i].bytes;
            a.at[a.n + 1] = a.at[a.n] + (segs[i].bytes + 15) / 16;
            ++a.n;
        }
        hipLaunchKernelGGL(pack_kernel, dim3(static_cast<unsigned>((units + 255) / 256)), dim3(256), 0,
                           st, a);
        check_hip(hipGetLastError(), "pack launch");
        check_hip(hipStreamSynchronize(st), "hipStreamSynchronize");
        int k = 0;
        for (size_t i = 0; i < nseg && !to_device; ++i) {
            if (!segs[i].bytes) continue;
            memcpy(segs[i].dst, a.dst[k++], segs[i].bytes);
        }
    } else {
        const size_t chunk_bytes = std::clamp(
            (total / (2 * copy_threads()) + 65535) & ~size_t(65535), kMinChunk, kChunk);
        // chunk c of the whole transfer: segment seg_of[c], offset off_of[c]
        std::vector<size_t> seg_of, off_of;
        for (size_t i = 0; i < nseg; ++i)
            for (size_t o = 0; o < segs[i].bytes; o += chunk_bytes) {
                seg_of.push_back(i);
                off_of.push_back(o);
            }
        const size_t nchunks = seg_of.size();
        const int nt = static_cast<int>(std::min<size_t>(copy_threads(), nchunks));
        Lanes taken(device, nt);
        auto& ls = taken.v;
        for (int t = 0; t < nt; ++t) ls[t]->init();

        std::atomic<size_t> next{0};
        std::atomic<bool> failed{false};
        std::mutex err_mu;
        std::string err;
        auto chunk = [&](size_t c, size_t* n) {
            const HostCopy& s = segs[seg_of[c]];
            *n = std::min(chunk_bytes, s.bytes - off_of[c]);
            return s;
        };
        // device -> host: the DMA of a lane's next chunk into one staging
        // buffer overlaps its memcpy of the other out to the destination
        auto to_host = [&](HostLane& ln) {
            size_t held[2];
            size_t bytes_of[2] = {0, 0};
            auto issue = [&](int b) -> bool {
                const size_t c = next.fetch_add(1);
                if (c >= nchunks || failed.load()) return false;
                size_t n;
                const HostCopy& s = chunk(c, &n);
                check_hip(hipMemcpyAsync(ln.stage[b], static_cast<const char*>(s.src) + off_of[c], n,
                                         hipMemcpyDeviceToHost, ln.stream),
                          "D2H stage");
                check_hip(hipEventRecord(ln.done[b], ln.stream), "hipEventRecord");
                held[b] = c;
                bytes_of[b] = n;
                return true;
            };
            bool more[2] = {issue(0), false};
            if (more[0]) more[1] = issue(1);
            int live = more[0] + more[1];
            for (int b = 0; live > 0; b ^= 1) {
                if (!more[b]) continue;
                check_hip(hipEventSynchronize(ln.done[b]), "hipEventSynchronize");
                const size_t c = held[b];
                memcpy(static_cast<char*>(segs[seg_of[c]].dst) + off_of[c], ln.stage[b], bytes_of[b]);
                more[b] = issue(b);
                if (!more[b]) --live;
            }
        };
        // host -> device: a lane fills one staging buffer while the DMA of
        // the other is in flight, waiting only before it refills a buffer
        auto to_dev = [&](HostLane& ln) {
            bool pending[2] = {false, false};
            for (int b = 0;; b ^= 1) {
                const size_t c = next.fetch_add(1);
                if (c >= nchunks || failed.load()) break;
                size_t n;
                const HostCopy& s = chunk(c, &n);
                if (pending[b]) check_hip(hipEventSynchronize(ln.done[b]), "hipEventSynchronize");
                memcpy(ln.stage[b], static_cast<const char*>(s.src) + off_of[c], n);
                check_hip(hipMemcpyAsync(static_cast<char*>(s.dst) + off_of[c], ln.stage[b], n,
                                         hipMemcpyHostToDevice, ln.stream),
                          "H2D stage");
                check_hip(hipEventRecord(ln.done[b], ln.stream), "hipEventRecord");
                pending[b] = true;
            }
            check_hip(hipStreamSynchronize(ln.stream), "hipStreamSynchronize");
        };
        auto worker = [&](int t) {
            HostLane& ln = *ls[t];
            try {
                check_hip(hipSetDevice(device), "hipSetDevice");
                if (to_device) to_dev(ln);
                else to_host(ln);
            } catch (const std::exception& ex) {
                failed.store(true);
                (void)hipStreamSynchronize(ln.stream);  // no DMA may outlive the call
                std::lock_guard<std::mutex> g(err_mu);
                if (err.empty()) err = ex.what();
            }
        };
        std::vector<std::thread> pool;
        pool.reserve(nt - 1);
        for (int t = 1; t < nt; ++t) pool.emplace_back(worker, t);
        worker(0);
        for (auto& th : pool) th.join();
        if (failed.load()) throw std::runtime_error("host copy: " + err);
    }
    const double ms =
        std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    if (!to_device && engine_order) {
        timings.handoff_ms = ms;
        timings.handoff_bytes = total;
    }
}

}  // namespace trw
