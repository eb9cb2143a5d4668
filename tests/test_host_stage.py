"""host_stage.h on the CPU under the thread sanitizer: the header compiled
against a stand-in for the few HIP calls it makes, whose stream is a thread
that runs copies and event records in order and late, so that a ring slot
refilled before its copy has left, or an unsynchronised hand-over between the
threads, is a reported race or a wrong byte."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#pragma once
#include <stddef.h>
#include <stdlib.h>
#include <string.h>
#include <condition_variable>
#include <deque>
#include <functional>
#include <mutex>
#include <thread>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum { hipMemcpyHostToDevice = 1, hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
struct Event { long due = 0; };
struct Stream {   // jobs in order on a thread of its own
    std::mutex m; std::condition_variable cv; std::deque<std::function<void()>> q;
    long queued = 0, done = 0; bool quit = false; int fail_after = -1;
    std::thread t{[this] {
        for (;;) {
            std::function<void()> f;
            { std::unique_lock<std::mutex> l(m); cv.wait(l, [&] { return quit || !q.empty(); }); if (q.empty()) return; f = q.front(); q.pop_front(); }
            std::this_thread::sleep_for(std::chrono::microseconds(300));
            f();
            { std::lock_guard<std::mutex> l(m); done++; }
            cv.notify_all();
        }
    }};
    void put(std::function<void()> f) { { std::lock_guard<std::mutex> l(m); q.push_back(f); queued++; } cv.notify_all(); }
    void wait(long n) { std::unique_lock<std::mutex> l(m); cv.wait(l, [&] { return done >= n; }); }
    ~Stream() { { std::lock_guard<std::mutex> l(m); quit = true; } cv.notify_all(); t.join(); }
};
using hipStream_t = Stream *;
using hipEvent_t = Event *;
inline Stream *&the_stream() { static Stream *s; return s; }
inline bool &no_pinned() { static bool b; return b; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, int) { if (no_pinned()) return hipErrorOutOfMemory; *p = malloc(n); return hipSuccess; }
inline hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, int) { *e = new Event; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t st) {
    if (st->fail_after >= 0 && st->fail_after-- == 0) return hipErrorUnknown;
    st->put([=] { memcpy(d, s, n); });
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { std::lock_guard<std::mutex> l(s->m); e->due = s->queued; return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t e) { the_stream()->wait(e->due); return hipSuccess; }
"""

MAIN = r"""
#include "host_stage.h"
#include <signal.h>
#include <stdio.h>
#include <unistd.h>
#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); _exit(3); } } while (0)
static pthread_t handled_on;
static void on_signal(int) { handled_on = pthread_self(); }
int main() {
    if (std::thread::hardware_concurrency() < HostStage::kThreads + 2) { puts("skipped"); return 0; }
    no_pinned() = true;
    CHECK(!HostStage::create());
    no_pinned() = false;
    sigset_t usr1;
    sigemptyset(&usr1);
    sigaddset(&usr1, SIGUSR1);
    signal(SIGUSR1, on_signal);
    pthread_sigmask(SIG_BLOCK, &usr1, nullptr);
    Stream s;                                        // (its thread never takes the signal)
    the_stream() = &s;
    pthread_sigmask(SIG_UNBLOCK, &usr1, nullptr);
    HostStage *h = HostStage::create();
    CHECK(h);
    sigset_t now;
    pthread_sigmask(SIG_BLOCK, &usr1, &now);         // the ring's threads alone could take it from here on
    CHECK(!sigismember(&now, SIGUSR1));              // the caller's mask is as it was
    // blobs that end inside slots and parts, more slots than the ring has, a copy that fails and
    // the run after it, the largest run
    const struct { int n; size_t bytes; int fail; } runs[] = {
        {1, 5, -1}, {1, HostStage::kSlot, -1}, {10, 3000001, -1}, {10, 9000000, 2}, {10, 8159232, -1}, {10, 12u << 20, -1}};
    uint32_t seed = 1;
    for (auto r : runs) {
        std::vector<std::vector<unsigned char>> src(r.n, std::vector<unsigned char>(r.bytes));
        std::vector<unsigned char> want, got(r.n * r.bytes);
        std::vector<void *> p;
        for (auto &b : src) {
            for (size_t i = 0; i < b.size(); i += 129) b[i] = (seed = seed * 1664525u + 1013904223u) >> 24;
            want.insert(want.end(), b.begin(), b.end());
            p.push_back(b.data());
        }
        s.fail_after = r.fail;
        const hipError_t e = h->run(p.data(), r.n, r.bytes, got.data(), &s);
        s.fail_after = -1;
        CHECK((e == hipSuccess) == (r.fail < 0));
        for (auto &b : src) memset(b.data(), 0xEE, b.size());   // every source byte has been read
        s.wait(s.queued);
        if (r.fail < 0) CHECK(got == want);
        kill(getpid(), SIGUSR1);
        printf("%d x %zu\n", r.n, r.bytes);
        fflush(stdout);
    }
    delete h;
    pthread_sigmask(SIG_UNBLOCK, &usr1, nullptr);
    CHECK(pthread_equal(handled_on, pthread_self()));
    puts("done");
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_ring_under_thread_sanitizer(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "ring"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=thread", "-pthread", f"-I{tmp_path}",
                        "-I" + os.path.join(ROOT, "fomoe_amd", "csrc"), str(tmp_path / "main.cpp"), "-o", str(exe)],
                       capture_output=True, text=True, timeout=300)
    if r.returncode and "libtsan" in r.stderr:
        pytest.skip("no thread sanitizer runtime")
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, TSAN_OPTIONS="halt_on_error=1:exitcode=66"))
    assert r.returncode == 0, r.stdout[-1000:] + r.stderr[-4000:]
    if "skipped" in r.stdout:
        pytest.skip("fewer CPUs than the ring's threads")
    assert "done" in r.stdout
