// host_lanes.hpp -- fields between device and host memory, in chunks through
// pinned buffers that the kernels write (or read) themselves.
//
// A copy into memory the caller has just allocated is bound by the first touch
// of its pages on the host (about 3 GB/s for one thread), not by the bus (55
// GB/s): several threads take the chunks of a large transfer in turn, each
// with two pinned buffers, so one fills while the other is copied out.
//
// A 128x96x80 FP32 domain's moments, state and flags to the host and its state
// back, 173 MB: 11.9 ms through a device staging buffer, 5.4 ms this way;
// velocity and density of 97x61x83 in FP64 after 21 steps: 1.46 -> 1.11 ms.
#pragma once

#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace lbm {

struct HostLane {
    static constexpr size_t kChunk = (size_t)2 << 20;
    char *buf[2] = {nullptr, nullptr};
    hipEvent_t ev[2] = {nullptr, nullptr};
    int device = 0;
};

// The process's lanes, at most kLanes (48 MB pinned), kept until release().
class HostLanes {
  public:
    static constexpr int kLanes = 12;
    static HostLanes &get() {
        static HostLanes *l = new HostLanes();  // outlives every transfer
        return *l;
    }
    // Up to `want` (<= kLanes) lanes on the current device `device`, at least one: waits
    // for one while every lane is in use (their holders need no further ones).
    // Empty: no memory for a single lane.
    std::vector<HostLane *> take(int device, int want) {
        std::vector<HostLane *> got;
        got.reserve(kLanes);
        std::unique_lock<std::mutex> lock(mutex_);
        for (;;) {
            for (size_t i = idle_.size(); i-- > 0 && (int)got.size() < want;)
                if (idle_[i]->device == device) {
                    got.push_back(idle_[i]);
                    idle_.erase(idle_.begin() + (long)i);
                }
            while ((int)got.size() < want && made_ < kLanes) {
                HostLane *l = make(device);
                if (!l) break;
                ++made_;
                got.push_back(l);
            }
            if (!got.empty()) return got;
            if (made_ == 0) return got;
            // every lane is busy, or idle ones belong to other devices
            if (!idle_.empty()) {
                destroy(idle_.back());
                idle_.pop_back();
                --made_;
                continue;
            }
            given_.wait(lock);
        }
    }
    void give(const std::vector<HostLane *> &lanes) {
        std::lock_guard<std::mutex> lock(mutex_);
        idle_.insert(idle_.end(), lanes.begin(), lanes.end());
        given_.notify_all();
    }
    // Frees the lanes that no transfer holds.
    void release() {
        std::lock_guard<std::mutex> lock(mutex_);
        for (HostLane *l : idle_) destroy(l);
        made_ -= (int)idle_.size();
        idle_.clear();
        given_.notify_all();  // one may be made now
    }

  private:
    HostLanes() { idle_.reserve(kLanes); }  // so giving back never allocates
    static HostLane *make(int device) {
        HostLane *l = new (std::nothrow) HostLane();
        if (!l) return nullptr;
        l->device = device;
        bool ok = true;
        for (int b = 0; b < 2; ++b) {
            ok = ok && hipHostMalloc((void **)&l->buf[b], HostLane::kChunk, hipHostMallocPortable) == hipSuccess;
            ok = ok && hipEventCreateWithFlags(&l->ev[b], hipEventDisableTiming) == hipSuccess;
        }
        if (ok) return l;
        (void)hipGetLastError();
        destroy(l);
        return nullptr;
    }
    static void destroy(HostLane *l) {
        for (int b = 0; b < 2; ++b) {
            if (l->buf[b]) (void)hipHostFree(l->buf[b]);
            if (l->ev[b]) (void)hipEventDestroy(l->ev[b]);
        }
        delete l;
    }
    std::mutex mutex_;
    std::condition_variable given_;
    std::vector<HostLane *> idle_;
    int made_ = 0;
};

// Moves the `comps` components of `n` cells, `elem` bytes each, between the
// host arrays host[i] (component i, n elements) and the device.
// launch(first, count, pinned) enqueues on `stream` the kernel that writes (or
// reads) `count` cells from cell `first` of every component to (from) `pinned`
// as [component][count].  Returns when all is done.  hipErrorOutOfMemory: no
// pinned memory.
template <bool OUT, class Launch>
hipError_t move_fields(int device, hipStream_t stream, long long n, int comps, size_t elem, char *const *host,
                       Launch &&launch) {
    // A launch adds about 16 us to a chunk's time on the bus (19 us a MB), small
    // chunks start the copies on the host sooner: 173 MB take 8.8 / 6.3 / 5.4 /
    // 5.8 ms in chunks of 0.5 / 1 / 2 / 4 MB, 13 MB 1.13 / 1.09 / 1.12 / 1.25 ms.
    // Into the device no fresh pages slow the host down, and the kernels' launches
    // count more: 4.9 MB take 0.23 / 0.16 ms in chunks of 1 / 2 MB, 8.4 MB 0.35 /
    // 0.29 (with a lane for each chunk; with one for two 0.31), 16 MB 0.58 / 0.47.
    // The runtime's own copy to a staging buffer on the device took 0.18, 0.28, 0.49.
    const size_t bytes = (size_t)n * (size_t)comps * elem;
    const bool large = bytes >= (size_t)(OUT ? 32 : 4) << 20;
    const size_t chunk = large ? HostLane::kChunk : HostLane::kChunk / 2;
    const long long per = (long long)(chunk / ((size_t)comps * elem)) / 64 * 64;
    const long long chunks = (n + per - 1) / per;
    // A thread costs about 30 us to start, a fresh megabyte up to 300 us; with 4
    // threads the 173 MB take 5.9 ms, with more than 6 what they take with 6.
    const int want = (int)std::max<long long>(1, std::min<long long>(6, !OUT && large ? chunks : chunks / 2));
    int before = device;  // the caller's device, current again when this returns
    if (hipGetDevice(&before) != hipSuccess) before = device;
    if (before != device) {
        const hipError_t e = hipSetDevice(device);
        if (e != hipSuccess) return e;
    }
    HostLanes &pool = HostLanes::get();
    std::vector<HostLane *> lanes;
    std::vector<std::thread> threads;
    try {
        threads.reserve((size_t)want);
        lanes = pool.take(device, want);
    } catch (const std::bad_alloc &) {
    }
    if (lanes.empty()) {
        if (before != device) (void)hipSetDevice(before);
        return hipErrorOutOfMemory;
    }
    const int W = (int)lanes.size();
    std::atomic<int> first_error{(int)hipSuccess};
    auto note = [&](hipError_t e) {
        int none = (int)hipSuccess;
        if (e != hipSuccess) first_error.compare_exchange_strong(none, (int)e);
        return e == hipSuccess;
    };
    auto copy = [&](long long c, char *buf) {
        const long long e0 = c * per, count = std::min(per, n - e0);
        for (int i = 0; i < comps; ++i) {
            char *h = host[i] + (size_t)e0 * elem, *p = buf + (size_t)i * count * elem;
            if (OUT) memcpy(h, p, (size_t)count * elem);
            else memcpy(p, h, (size_t)count * elem);
        }
    };
    auto issue = [&](long long c, HostLane *l, int b) {
        const long long e0 = c * per;
        if (!note(launch(e0, std::min(per, n - e0), (void *)l->buf[b]))) return false;
        if (note(hipEventRecord(l->ev[b], stream))) return true;
        (void)hipStreamSynchronize(stream);  // the kernel may still use the buffer
        return false;
    };
    auto work = [&](int t) {
        HostLane *l = lanes[(size_t)t];
        if (t > 0 && !note(hipSetDevice(device))) return;  // 0 is the caller's own thread
        int b = 0;
        bool pending[2] = {false, false};
        if (OUT) {
            for (int q = 0; q < 2; ++q)
                if (t + (long long)q * W < chunks) pending[q] = issue(t + (long long)q * W, l, q);
            for (long long c = t; c < chunks && pending[b]; c += W, b ^= 1) {
                pending[b] = false;
                if (!note(hipEventSynchronize(l->ev[b]))) break;
                copy(c, l->buf[b]);
                if (c + 2LL * W < chunks) pending[b] = issue(c + 2LL * W, l, b);
            }
        } else {
            for (long long c = t; c < chunks; c += W, b ^= 1) {
                if (pending[b] && !note(hipEventSynchronize(l->ev[b]))) break;
                copy(c, l->buf[b]);
                pending[b] = issue(c, l, b);
                if (!pending[b]) break;
            }
        }
        for (int q = 0; q < 2; ++q)  // nothing uses the lane any more when it goes back
            if (pending[q]) note(hipEventSynchronize(l->ev[q]));
    };
    // Wait for the work before the transfer once, not in every thread.
    if (W > 1) note(hipStreamSynchronize(stream));
    int started = 1;
    try {
        for (; started < W; ++started) threads.emplace_back(work, started);
    } catch (...) {
        // no more threads: their chunks are done here
    }
    work(0);
    for (int t = started; t < W; ++t) work(t);
    for (std::thread &t : threads) t.join();
    pool.give(lanes);
    if (before != device) (void)hipSetDevice(before);
    return (hipError_t)first_error.load();
}

}  // namespace lbm
