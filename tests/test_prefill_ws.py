"""prefill_ws.h on the CPU: the header compiled against a stand-in device with
a limited memory. Which pass sizes a call gets, that a card with little room
is left half of it, and that the calls after the first neither allocate nor
free nor wait, also where the device refuses what it said was free."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = """
#pragma once
#include <stddef.h>
#include <stdint.h>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
"""

MAIN = r"""
#include "prefill_ws.h"
#include <array>
#include <map>
#include <stdio.h>
#include <stdlib.h>
#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); exit(3); } } while (0)
struct Dev {
    size_t size, told = 0;               // told: what it says is free beyond that
    hipError_t error = hipErrorOutOfMemory;
    size_t used = 0, peak = 0;
    int allocs = 0, frees = 0, waits = 0;
    std::map<void *, size_t> held;
    hipError_t alloc(void **p, size_t n) {
        allocs++;
        *p = nullptr;
        if (used + n > size) return error;
        *p = malloc(1);
        held[*p] = n;
        used += n;
        peak = used > peak ? used : peak;
        return hipSuccess;
    }
    void free(void *p) { CHECK(held.count(p)); frees++; used -= held[p]; held.erase(p); ::free(p); }
    hipError_t wait() { waits++; return hipSuccess; }
    size_t free_bytes() { return size + told - used; }
    int calls() const { return allocs + frees + waits; }
};
struct Ctx {                             // 100 bytes of a call's token, 1000 and 3000 of a pass's
    std::array<void *, 3> p{};
    std::array<size_t, 3> cap{};
    size_t refused = SIZE_MAX;
    hipError_t fit(Dev &d, int T, int most, int chunk, int &Tc) {
        return fo::prefill_fit(d, T, most, chunk, refused, [&](int t) {
            return std::array<fo::PfBuf, 3>{fo::PfBuf{&p[0], &cap[0], (size_t)T * 100},
                                            fo::PfBuf{&p[1], &cap[1], (size_t)t * 1000},
                                            fo::PfBuf{&p[2], &cap[2], (size_t)t * 3000}}; }, Tc);
    }
    bool holds(int T, int Tc) { return cap[0] >= (size_t)T * 100 && cap[1] >= (size_t)Tc * 1000 && cap[2] >= (size_t)Tc * 3000; }
};
int main() {
    // passes: as few as `most` allows, equal, whole chunks
    for (int chunk : {32, 1024, 5216})
        for (int n : {1, 7, 11}) {
            const int most = n * chunk;
            for (int T : {1, chunk - 1, chunk, chunk + 1, most - 1, most, most + 1, 2 * most, 2 * most + 1, 5 * most + 7}) {
                const int Tc = fo::prefill_even_pass(T, most, chunk);
                CHECK(Tc >= 1 && Tc <= most && (Tc == T || Tc % chunk == 0));
                CHECK((T + Tc - 1) / Tc == (T + most - 1) / most);
                CHECK(T <= most ? Tc == T : (T + Tc - 1) / Tc * (Tc - chunk) < T);   // one chunk less takes more passes
            }
        }
    int Tc;
    {   // room for everything; a second call, a shorter one, a longer one
        Dev d{1000000000};
        Ctx c;
        CHECK(c.fit(d, 10000, 11264, 1024, Tc) == hipSuccess && Tc == 10000 && c.holds(10000, Tc));
        int n = d.calls();
        CHECK(n == 3);
        CHECK(c.fit(d, 10000, 11264, 1024, Tc) == hipSuccess && Tc == 10000 && d.calls() == n);
        CHECK(c.fit(d, 16, 11264, 1024, Tc) == hipSuccess && Tc == 16 && d.calls() == n);
        CHECK(c.fit(d, 11265, 11264, 1024, Tc) == hipSuccess && Tc == 6144 && c.holds(11265, Tc));
        CHECK(d.waits == 0);
    }
    {   // little room: at most half of what is free, and nothing more once held
        Dev d{32000000};
        Ctx c;
        CHECK(c.fit(d, 10000, 11264, 1024, Tc) == hipSuccess && Tc == 2048 && c.holds(10000, Tc));
        CHECK(d.peak <= d.size / 2 && d.waits == 0 && d.frees == 0);
        const int n = d.calls();
        for (int i = 0; i < 3; i++) CHECK(c.fit(d, 10000, 11264, 1024, Tc) == hipSuccess && Tc == 2048 && d.calls() == n);
        d.size = 1000000000;              // the card empties: the full pass again
        CHECK(c.fit(d, 10000, 11264, 1024, Tc) == hipSuccess && Tc == 10000);
    }
    {   // one chunk is asked for whatever is free; what the device refuses there is the call's error
        Dev d{6000000};
        Ctx c;
        CHECK(c.fit(d, 10000, 11264, 1024, Tc) == hipSuccess && Tc == 1024 && c.holds(10000, Tc));
        Dev e{5000000};
        Ctx f;
        CHECK(f.fit(e, 10000, 11264, 1024, Tc) == hipErrorOutOfMemory && f.refused == SIZE_MAX);
        CHECK(f.fit(e, 700, 11264, 1024, Tc) == hipSuccess && Tc == 700 && f.holds(700, 700));
    }
    {   // refused though said to be free: given back, then smaller, and not tried again
        Dev d{20000000};
        d.told = 1000000000;
        Ctx c;
        CHECK(c.fit(d, 10000, 11264, 1024, Tc) == hipSuccess && c.holds(10000, Tc) && Tc == 2048 && d.waits > 0);
        const int n = d.calls();
        for (int i = 0; i < 3; i++) CHECK(c.fit(d, 10000, 11264, 1024, Tc) == hipSuccess && Tc == 2048 && d.calls() == n);
    }
    {   // any other error is the call's
        Dev d{20000000};
        d.told = 1000000000;
        d.error = hipErrorUnknown;
        Ctx c;
        CHECK(c.fit(d, 10000, 11264, 1024, Tc) == hipErrorUnknown && d.waits == 0);
    }
    puts("done");
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_prefill_workspace(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "ws"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", f"-I{tmp_path}", "-I" + os.path.join(ROOT, "fomoe_amd", "csrc"),
                        str(tmp_path / "main.cpp"), "-o", str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "done" in r.stdout, r.stdout[-1000:] + r.stderr[-2000:]
