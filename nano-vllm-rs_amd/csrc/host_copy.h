// host_copy.h — large device arrays into a program's own (pageable) memory.
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace nvr {

// The runtime copies to pageable memory through one staging buffer and one thread, which also takes the page faults of an array that was just allocated: 39 MB of logits of 64 sequences 3.9 ms, of
// which the link needs 0.8.  Here LANES threads (the caller and three that live for the call) each bring every LANES-th piece into two pinned pieces in turn, on the stream that the array is made on,
// and copy one to its place while the other lands: 1.5 ms.  (A stream for each thread is no faster, and its first use takes a millisecond.)  Nothing outlives a call but the pinned pieces (8 MiB a
// runner, a millisecond of the eleven that it takes to be made); calls on one object take turns.
class HostCopy {
public:
    static constexpr size_t PIECE = 1 << 20, LEAST = 8 << 20;              // (LEAST: below, the runtime's own copy is as fast)
    static constexpr int LANES = 4;
    ~HostCopy() { release(); }
    // Once, on the device's thread; not within a capture.  Where the pieces or an event are not to be had nothing is kept, and the runtime copies (takes)
    void prepare() {
        if (pinned) return;
        hipError_t e = hipHostMalloc((void **)&pinned, PIECE * 2 * LANES, hipHostMallocDefault);
        if (e != hipSuccess) pinned = nullptr;
        for (int t = 0; t < LANES; ++t) {
            lanes[t].at = pinned ? pinned + (size_t)t * 2 * PIECE : nullptr;
            for (int i = 0; i < 2 && e == hipSuccess; ++i)
                if ((e = hipEventCreateWithFlags(&lanes[t].landed[i], hipEventDisableTiming)) != hipSuccess) lanes[t].landed[i] = nullptr;
        }
        if (e != hipSuccess) { release(); (void)hipGetLastError(); }
    }
    // whether `to` is memory that this copies to: neither the runtime's own (pinned, managed or device memory, which it copies to at the link's rate) nor too little
    bool takes(const void *to, size_t bytes) const {
        if (!pinned || bytes < LEAST) return false;
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, to) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
        (void)hipGetLastError();
        return true;
    }
    // `from` as it is behind the work that is on `stream` now; the call ends when `to` is complete
    hipError_t run(int device, hipStream_t stream, void *to, const void *from, size_t bytes) {
        std::lock_guard<std::mutex> turn(busy);
        hipError_t rc[LANES] = {};
        std::vector<std::thread> threads;
        int started = 1;
        try {
            threads.reserve(LANES - 1);
            for (; started < LANES; ++started) threads.emplace_back([this, &rc, device, stream, to, from, bytes, t = started] { rc[t] = lane(t, device, stream, (char *)to, (const char *)from, bytes); });
        } catch (...) {}                                                   // (no thread to be had: the caller takes their pieces too)
        rc[0] = lane(0, device, stream, (char *)to, (const char *)from, bytes);
        for (int t = started; t < LANES; ++t) rc[t] = lane(t, device, stream, (char *)to, (const char *)from, bytes);
        for (std::thread &t : threads) t.join();
        for (hipError_t e : rc) if (e != hipSuccess) return e;
        return hipSuccess;
    }

private:
    struct Lane { char *at = nullptr; hipEvent_t landed[2] = {}; } lanes[LANES];
    char *pinned = nullptr;
    std::mutex busy;
    void release() {
        for (Lane &l : lanes)
            for (hipEvent_t &e : l.landed) if (e) { (void)hipEventDestroy(e); e = nullptr; }
        if (pinned) (void)hipHostFree(pinned);
        pinned = nullptr;
    }
    hipError_t lane(int t, int device, hipStream_t stream, char *to, const char *from, size_t bytes) {
        const Lane &l = lanes[t];
        if (hipError_t e = hipSetDevice(device)) return e;
        const size_t pieces = (bytes + PIECE - 1) / PIECE;
        auto size = [&](size_t p) { return std::min(PIECE, bytes - p * PIECE); };
        auto request = [&](size_t p, int slot) {
            if (hipError_t e = hipMemcpyAsync(l.at + slot * PIECE, from + p * PIECE, size(p), hipMemcpyDeviceToHost, stream)) return e;
            return hipEventRecord(l.landed[slot], stream);
        };
        hipError_t e = hipSuccess;
        int slot = 0;
        if ((size_t)t < pieces) e = request(t, 0);
        for (size_t p = t; e == hipSuccess && p < pieces; p += LANES, slot ^= 1) {
            if (p + LANES < pieces) e = request(p + LANES, slot ^ 1);
            if (e == hipSuccess) e = hipEventSynchronize(l.landed[slot]);
            if (e == hipSuccess) std::memcpy(to + p * PIECE, l.at + slot * PIECE, size(p));
        }
        if (e != hipSuccess) (void)hipStreamSynchronize(stream);         // (nothing is left under way into the pinned pieces)
        return e;
    }
};

}  // namespace nvr
