// jw_host.hpp -- transfers between caller's (pageable) memory and the device.
//
// A transfer is cut into chunks; lane w takes chunks w, w + L, ...: the kernel that converts
// the chunk on its way (field planes to AoS, a real part, ...) works on the lane's
// pinned buffer across the bus, and a host thread copies between that buffer and the
// caller's memory.  What bounds it is the host side: a fresh destination's page faults
// and one thread's copy (38 MB into fresh pages: 8.2 ms by one thread, 3.0 by four, and
// 3.0 and 0.8 in huge pages, against 0.7 on the bus; the runtime's own pageable copy takes
// 9.7).  L = 4; one lane, without threads, below 1 MiB, where starting them costs more.
//
// A pinned buffer costs 32 us to allocate and 18 to free, a call at N = 64 that uses one saves 10.
// So a context's first kStagedCalls transfers below kStagedBelow go through a device buffer
// (under 2 us to allocate up to 1 MiB) and the runtime's copy, as all do when no pinned memory
// is to be had.  us of a fresh context's first upload and download, with four lanes
// allocated at once / staged: N = 4 83, 83 / 20, 29; 64 134, 129 / 46, 51; 128 219, 239 / 127, 173.
#pragma once

#include "jw_internal.hpp"

#include <string.h>

#include <thread>

namespace jw {

constexpr size_t kLaneBytes = (size_t)4 << 20;      // largest chunk
constexpr size_t kLanesFrom = (size_t)1 << 20;      // transfers from here on use all lanes
constexpr size_t kStageBytes = (size_t)1 << 20;     // largest chunk through the device buffer
constexpr size_t kStagedBelow = (size_t)4 << 20;
constexpr int kStagedCalls = 4;

inline void lane_free(jw_ctx* c, int w) {
    if (c->lane_pin[w]) (void)hipHostFree(c->lane_pin[w]);
    if (c->lane_ev[w]) (void)hipEventDestroy(c->lane_ev[w]);
    c->lane_pin[w] = nullptr;
    c->lane_ev[w] = nullptr;
    c->lane_cap[w] = 0;
}

inline void staging_free(jw_ctx* c) {
    for (int w = 0; w < JW_LANES; w++) lane_free(c, w);
    if (c->stage) (void)hipFree(c->stage);
    c->stage = nullptr;
    c->stage_cap = 0;
}

// lanes 0 .. lanes - 1 of at least `bytes` each (no work is pending on them: every
// transfer waits for its own)
inline hipError_t lanes_ensure(jw_ctx* c, int lanes, size_t bytes) {
    for (int w = 0; w < lanes; w++) {
        if (c->lane_cap[w] >= bytes) continue;
        lane_free(c, w);
        // coherent: a kernel's stores are the host's to see once its event is through
        hipError_t e = hipHostMalloc(&c->lane_pin[w], bytes, hipHostMallocCoherent);
        if (e == hipSuccess)
            e = hipEventCreateWithFlags(&c->lane_ev[w], hipEventDisableTiming | hipEventReleaseToSystem);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            lane_free(c, w);
            return e;
        }
        c->lane_cap[w] = bytes;
    }
    return hipSuccess;
}

// the transfer through the device buffer, a chunk at a time: the runtime copies between
// it and the caller's memory
template <typename F>
inline hipError_t staged_transfer(jw_ctx* c, void* host, size_t items, size_t size, bool to_host, F&& launch) {
    const size_t most = kStageBytes / size ? kStageBytes / size : 1, per = items < most ? items : most;
    hipError_t e = hipSuccess;
    if (c->stage_cap < per * size) {
        if (c->stage) (void)hipFree(c->stage);
        c->stage = nullptr;
        c->stage_cap = 0;
        if ((e = hipMalloc(&c->stage, per * size)) != hipSuccess) {
            (void)hipGetLastError();
            return e;
        }
        c->stage_cap = per * size;
    }
    for (size_t first = 0; first < items && e == hipSuccess; first += per) {
        const size_t n = items - first < per ? items - first : per;
        char* const h = static_cast<char*>(host) + first * size;
        if (!to_host) e = hipMemcpyAsync(c->stage, h, n * size, hipMemcpyHostToDevice, c->stream);
        if (e == hipSuccess) e = launch(c->stage, first, n);
        if (to_host && e == hipSuccess) e = hipMemcpyAsync(h, c->stage, n * size, hipMemcpyDeviceToHost, c->stream);
    }
    const hipError_t s = hipStreamSynchronize(c->stream);
    return e != hipSuccess ? e : s;
}

// items of `size` bytes between host and device; to_host: launch(buf, first, n) fills the
// buffer with items first .. first + n - 1, else it takes them from it.  Returns
// when the caller's memory is written, or may be reused.
template <typename F>
inline hipError_t host_transfer(jw_ctx* c, void* host, size_t items, size_t size, bool to_host, F&& launch) {
    // the calling thread's current device is left as it was
    struct OnDevice {
        int was = 0;
        hipError_t e;
        explicit OnDevice(int d) {
            e = hipGetDevice(&was);
            if (e == hipSuccess && was != d) e = hipSetDevice(d);
        }
        ~OnDevice() { (void)hipSetDevice(was); }
    } dev(c->device);
    if (dev.e != hipSuccess) return dev.e;
    const size_t total = items * size;
    const int lanes = total >= kLanesFrom ? JW_LANES : 1;
    size_t per = (items + lanes - 1) / lanes;                       // items of a chunk
    const size_t most = kLaneBytes / size ? kLaneBytes / size : 1;
    if (per > most) per = most;
    if (total < kStagedBelow && c->staged < kStagedCalls) {
        c->staged++;
        if (staged_transfer(c, host, items, size, to_host, launch) == hipSuccess) return hipSuccess;
    }
    hipError_t e = lanes_ensure(c, lanes, per * size);
    if (e != hipSuccess) return staged_transfer(c, host, items, size, to_host, launch);
    const size_t chunks = (items + per - 1) / per;
    hipError_t res[JW_LANES] = {};
    auto lane = [&](int w) {
        hipError_t r = hipSetDevice(c->device);
        char* const pin = static_cast<char*>(c->lane_pin[w]);
        for (size_t k = w; k < chunks && r == hipSuccess; k += lanes) {
            const size_t first = k * per, n = items - first < per ? items - first : per;
            char* const h = static_cast<char*>(host) + first * size;
            if (!to_host) {
                if (k >= (size_t)lanes) r = hipEventSynchronize(c->lane_ev[w]);      // the buffer's last chunk is taken
                memcpy(pin, h, n * size);
            }
            if (r == hipSuccess) r = launch(pin, first, n);
            if (r == hipSuccess) r = hipEventRecord(c->lane_ev[w], c->stream);
            if (to_host && r == hipSuccess) {
                r = hipEventSynchronize(c->lane_ev[w]);
                if (r == hipSuccess) memcpy(h, pin, n * size);
            }
        }
        res[w] = r;
    };
    std::thread th[JW_LANES];
    for (int w = 1; w < lanes; w++) {
        try {
            th[w] = std::thread(lane, w);
        } catch (...) {      // no thread to be had: the caller's runs the lane below
        }
    }
    lane(0);
    for (int w = 1; w < lanes; w++) {
        if (th[w].joinable()) th[w].join();
        else lane(w);
    }
    // whatever happened, nothing is left running on the buffers
    const hipError_t s = hipStreamSynchronize(c->stream);
    for (int w = 0; w < lanes; w++)
        if (res[w] != hipSuccess) return res[w];
    return s;
}

}  // namespace jw
