"""csrc/host_copy.h on the CPU, over a stand-in for the runtime whose copies are made by a thread of its own: pieces or events that are not to be had, and several callers at once.  Built with the
thread sanitizer (a race ends the program) and run here."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = r"""
#pragma once
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <thread>
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2, hipMemcpyDeviceToHost = 2 };
struct hipPointerAttribute_t { hipMemoryType type; };
struct Stream {                                            // works through what it is given in order, on its own thread
    std::mutex m; std::condition_variable cv; std::deque<std::function<void()>> q; bool busy = false, end = false; std::thread t;
    Stream() : t([this] { for (;;) { std::unique_lock<std::mutex> l(m); cv.wait(l, [&] { return end || !q.empty(); }); if (q.empty()) return; auto f = q.front(); q.pop_front(); busy = true; l.unlock(); f(); l.lock(); busy = false; cv.notify_all(); } }) {}
    ~Stream() { { std::lock_guard<std::mutex> l(m); end = true; } cv.notify_all(); t.join(); }
    void push(std::function<void()> f) { { std::lock_guard<std::mutex> l(m); q.push_back(f); } cv.notify_all(); }
    void wait() { std::unique_lock<std::mutex> l(m); cv.wait(l, [&] { return q.empty() && !busy; }); }
};
struct Event { std::mutex m; std::condition_variable cv; long asked = 0, done = 0; };
typedef Stream *hipStream_t;
typedef Event *hipEvent_t;
inline std::atomic<int> live_hosts{0}, live_events{0}, copies{0}, calls{0}, failing{-1}, failing_copy{-1};      // failing: number of the call that fails
inline hipError_t last = hipSuccess;
inline hipError_t give(hipError_t e) { if (e) last = e; return e; }
inline hipError_t hipGetLastError() { hipError_t e = last; last = hipSuccess; return e; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) { if (calls++ == failing) return give(hipErrorOutOfMemory); *p = malloc(n); ++live_hosts; return hipSuccess; }
inline hipError_t hipHostFree(void *p) { free(p); --live_hosts; return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { if (calls++ == failing) return give(hipErrorOutOfMemory); *e = new Event; ++live_events; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; --live_events; return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return give(hipErrorInvalidValue); }      // (memory that the runtime does not know)
inline hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, int, hipStream_t s) { if (copies++ == failing_copy) return hipErrorInvalidValue; s->push([=] { std::memcpy(to, from, n); }); return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { long n; { std::lock_guard<std::mutex> l(e->m); n = ++e->asked; } s->push([=] { { std::lock_guard<std::mutex> l(e->m); e->done = n; e->cv.notify_all(); } }); return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t e) { std::unique_lock<std::mutex> l(e->m); const long n = e->asked; e->cv.wait(l, [&] { return e->done >= n; }); return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t s) { s->wait(); return hipSuccess; }
"""

PROGRAM = r"""
#include "host_copy.h"
#include <cstdio>
#define EXPECT(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
    using nvr::HostCopy;
    const size_t bytes = 9 * HostCopy::PIECE + 4096 + 12;
    std::vector<char> from(bytes), to(bytes), other(bytes);
    for (size_t i = 0; i < bytes; ++i) from[i] = (char)(i * 2654435761u >> 24);
    Stream s;
    for (int n = 0; n < 1 + 2 * HostCopy::LANES; ++n) {                    // each call of the preparation fails once: nothing is kept, no error is left behind, and nothing is taken
        failing = n; calls = 0;
        HostCopy c;
        c.prepare();
        EXPECT(calls > n && live_hosts == 0 && live_events == 0 && hipGetLastError() == hipSuccess && !c.takes(to.data(), bytes));
        failing = -1;
        c.prepare();                                                  // (and a later attempt finds an object that is as new)
        EXPECT(c.takes(to.data(), bytes) && hipGetLastError() == hipSuccess);
    }
    EXPECT(live_hosts == 0 && live_events == 0);
    {
        HostCopy c;
        EXPECT(!c.takes(to.data(), bytes));                                // (not prepared)
        c.prepare();
        EXPECT(live_hosts == 1 && live_events == 2 * HostCopy::LANES && !c.takes(to.data(), HostCopy::LEAST - 1));
        for (size_t n : {bytes, (size_t)HostCopy::LEAST, 2 * HostCopy::PIECE + 4}) {      // (the last: fewer pieces than lanes)
            std::fill(to.begin(), to.end(), 0);
            EXPECT(c.run(0, &s, to.data(), from.data(), n) == hipSuccess && std::memcmp(to.data(), from.data(), n) == 0);
            EXPECT(n == bytes || to[n] == 0);
        }
        std::fill(to.begin(), to.end(), 0);
        hipError_t rc[2];
        std::thread second([&] { for (int i = 0; i < 3; ++i) rc[1] = c.run(0, &s, other.data(), from.data(), bytes); });
        for (int i = 0; i < 3; ++i) rc[0] = c.run(0, &s, to.data(), from.data(), bytes);
        second.join();
        EXPECT(rc[0] == hipSuccess && rc[1] == hipSuccess && to == from && other == from);
        for (int n = 0; n < 10; ++n) {                                     // a request that is refused: the call says so, and nothing is under way behind it
            copies = 0; failing_copy = n;
            EXPECT(c.run(0, &s, to.data(), from.data(), bytes) == hipErrorInvalidValue);
        }
        failing_copy = -1;
        std::fill(to.begin(), to.end(), 0);
        EXPECT(c.run(0, &s, to.data(), from.data(), bytes) == hipSuccess && to == from);
    }
    EXPECT(live_hosts == 0 && live_events == 0);
    std::puts("host copy ok");
}
"""


@pytest.mark.parametrize("sanitizer", ["thread", "address,undefined"])
def test_copy_and_its_preparation(tmp_path, sanitizer):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (tmp_path / "main.cpp").write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", f"-fsanitize={sanitizer}", "-I", str(tmp_path), "-I", os.path.join(ROOT, "nano-vllm-rs_amd", "csrc"), "-o", str(tmp_path / "main"),
                           str(tmp_path / "main.cpp"), "-pthread"])
    r = subprocess.run([str(tmp_path / "main")], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=120)
    assert r.returncode == 0 and "host copy ok" in r.stdout, (r.stdout[-500:], r.stderr[-2000:])
