// prefill_ws.h — how many tokens a prefill pass takes, and the workspace for it.
//
// The workspace is the context's and only grows. One chunk's is always asked
// for. A larger pass is a matter of speed alone (a pass reads the weights
// once; the output bits are the same), so it grows the workspace by at most
// half of the device's free memory: the rest stays the program's. On a full
// card the passes are those that the held workspace takes, call after call,
// and nothing is allocated, given back or waited for.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace fo {

struct PfBuf {
    void **p;
    size_t *cap;
    size_t need;
};

// Tokens per pass of T tokens, whole chunks and at most `most`: as few passes
// as that takes, of equal size.
inline int prefill_even_pass(int T, int most, int chunk) {
    if (T <= most) return T;
    const int c = (T + chunk - 1) / chunk, n = (T + most - 1) / most;
    return (c + n - 1) / n * chunk;
}

// Tc = the tokens of a pass (at most `most`), its workspace held. sizes(Tc)
// gives the buffers (a std::array of PfBuf); dev allocates, frees, waits for
// the work that may use them and knows the free memory. refused: the smallest
// workspace the device had no memory for after all, kept by the context and
// not tried again.
template <class Dev, class Sizes>
hipError_t prefill_fit(Dev &dev, int T, int most, int chunk, size_t &refused, Sizes sizes, int &Tc) {
    size_t room = 0;
    for (bool asked = false;;) {
        Tc = prefill_even_pass(T, most, chunk);
        size_t total = 0, growth = 0;
        auto bufs = sizes(Tc);
        for (PfBuf &b : bufs) {
            total += b.need;
            growth += b.need > *b.cap ? b.need - *b.cap : 0;
        }
        if (!growth) return hipSuccess;
        const bool least = Tc <= chunk;
        if (!least && !asked) {
            room = dev.free_bytes() / 2;
            asked = true;
        }
        if (least || (growth <= room && total < refused)) {
            hipError_t e = hipSuccess;
            for (PfBuf &b : bufs) {
                if (*b.cap >= b.need) continue;
                if (*b.p) dev.free(*b.p);
                *b.p = nullptr;
                *b.cap = 0;
                e = dev.alloc(b.p, b.need);
                if (e != hipSuccess) break;
                *b.cap = b.need;
            }
            if (e != hipErrorOutOfMemory || least) return e;
            refused = total;
            e = dev.wait();
            if (e != hipSuccess) return e;
            for (PfBuf &b : bufs) {
                if (*b.p) dev.free(*b.p);
                *b.p = nullptr;
                *b.cap = 0;
            }
            room = dev.free_bytes() / 2;
        }
        const int half = (Tc + chunk - 1) / chunk / 2;
        most = (half > 1 ? half : 1) * chunk;
    }
}

}  // namespace fo
