// Read-back of context state to caller memory through pinned staging.
//
// What bounds a read-back of ordinary (pageable) caller memory is the host
// side: one thread copying through the driver's staging, page faults of fresh
// destination pages, and, for sphere scenes, the scatter from sorted slots to
// particle ids. Here kernels put the rows into the caller's layout and write
// them straight into pinned slots over the host link (coalesced stores), and
// several host threads, each owning two slots, copy them out while the next
// chunks are in flight.
#pragma once

#include <algorithm>
#include <atomic>
#include <mutex>
#include <thread>
#include <vector>

#include "sd_internal.hpp"

namespace sd {

// Pinned staging of one context, grown on demand, given back with the
// context's buffers. At most READBACK_THREADS * 2 slots.
struct HostStage {
    char* p = nullptr;
    size_t bytes = 0;
    std::mutex lock;  // read-backs of one context by several host threads take turns
    HostStage() = default;
    HostStage& operator=(const HostStage&) { return *this; }  // a context reset keeps its (released) staging
};
void stage_release(HostStage& st);
sd_status stage_reserve(HostStage& st, size_t bytes);

// Six threads: the copies of one thread, page faults included, run at a few
// GB/s, a sixth of what the link delivers.
constexpr int READBACK_THREADS = 6;

// Runs chunks 0 .. chunks-1: fill(chunk, slot, stream) enqueues the device work
// that writes the chunk into a slot, drain(chunk, slot) copies it out on the
// host once that work has ended. One chunk: no threads, no events.
template <typename Fill, typename Drain>
sd_status staged_chunks(HostStage& st, int chunks, size_t slot_bytes, hipStream_t s, Fill fill, Drain drain) {
    if (chunks <= 0) return SD_OK;
    if (chunks == 1) {
        sd_status e = stage_reserve(st, slot_bytes);
        if (e == SD_OK) e = fill(0, st.p, s);
        if (e != SD_OK) return e;
        SD_HIP(hipStreamSynchronize(s));
        drain(0, st.p);
        return SD_OK;
    }
    const int T = std::min(READBACK_THREADS, (chunks + 1) / 2);
    sd_status e = stage_reserve(st, slot_bytes * 2 * (size_t)T);
    if (e != SD_OK) return e;
    int dev = 0;
    SD_HIP(hipGetDevice(&dev));
    hipEvent_t ev[2 * READBACK_THREADS] = {};
    for (int k = 0; k < 2 * T && e == SD_OK; ++k)
        if (hipEventCreateWithFlags(&ev[k], hipEventDisableTiming) != hipSuccess)
            e = set_error(SD_ERR_HIP, "read-back: event creation failed");
    std::atomic<int> failed{0};
    auto work = [&](int t) {
        if (hipSetDevice(dev) != hipSuccess) {
            failed = 1;
            return;
        }
        auto start = [&](int c, int k) {
            if (fill(c, st.p + (size_t)(2 * t + k) * slot_bytes, s) != SD_OK ||
                hipEventRecord(ev[2 * t + k], s) != hipSuccess)
                failed = 1;
        };
        int k = 0;
        if (t < chunks) start(t, 0);
        for (int c = t; c < chunks && !failed; c += T, k ^= 1) {
            if (c + T < chunks) start(c + T, k ^ 1);  // (that slot was drained a turn ago)
            if (failed || hipEventSynchronize(ev[2 * t + k]) != hipSuccess) {
                failed = 1;
                break;
            }
            drain(c, st.p + (size_t)(2 * t + k) * slot_bytes);
        }
    };
    if (e == SD_OK) {
        std::thread th[READBACK_THREADS];
        bool own[READBACK_THREADS] = {};
        for (int t = 1; t < T; ++t) {
            try {
                th[t] = std::thread(work, t);
                own[t] = true;
            } catch (...) {  // no thread to be had: this one does its share below
            }
        }
        work(0);
        for (int t = 1; t < T; ++t) {
            if (own[t]) th[t].join();
            else work(t);
        }
    }
    // the staging and the caller's memory stay untouched after the return
    if (hipStreamSynchronize(s) != hipSuccess) failed = 1;
    for (hipEvent_t v : ev)
        if (v) (void)hipEventDestroy(v);
    if (e == SD_OK && failed) e = set_error(SD_ERR_HIP, "read-back failed: %s", hipGetErrorString(hipGetLastError()));
    return e;
}

// Sphere state by particle id: out[0..8] = x, y, z, vx, vy, vz, wx, wy, wz
// (n floats each, host, any may be NULL) from the rows of sorted slots. inv:
// n ints of device scratch.
sd_status readback_spheres(HostStage& st, const float4* pos, const float4* vel, const float4* omg, const int* ids,
                           int n, int* inv, float* const out[9], hipStream_t s);
}  // namespace sd
