// Host loops of the C ABI.  Plain C++.
#pragma once
#include <algorithm>
#include <atomic>
#include <cstdint>
#include <thread>
#include <vector>

namespace {

// Host loops over columns or rows run on up to 16 threads, fewer where no more can
// be started: each element is computed as in a serial loop, and the only
// reductions (a maximum, counts) do not depend on the order.
inline unsigned host_threads() {
    static const unsigned n = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
    return n;
}
template <class Fn>
void par_for(long lo, long hi, Fn fn) {            // fn(t, a, b): thread t covers [a, b)
    const long n = hi - lo;
    if (n <= 0) return;
    const long T = std::min<long>(host_threads(), n);
    if (T <= 1) { fn(0, lo, hi); return; }
    const long chunk = (n + T - 1) / T;
    std::vector<std::thread> th;
    long t = 1;
    auto from = [&](long q) { return std::min(hi, lo + q * chunk); };
    try {
        th.reserve((size_t)T - 1);
        for (; t < T && from(t) < hi; ++t) th.emplace_back(fn, (int)t, from(t), from(t + 1));
    } catch (...) {                                // no further thread: its part and the rest here
    }
    fn(0, lo, from(1));
    for (; t < T && from(t) < hi; ++t) fn((int)t, from(t), from(t + 1));
    for (auto &x : th) x.join();
}
// the first of n particles outside the cells 1..nii x 1..njj; n if there is none
inline int32_t first_outside(int32_t n, const int32_t *cell_i, const int32_t *cell_j, int nii, int njj) {
    std::atomic<int32_t> bad{n};
    par_for(0, ((long)n + 65535) / 65536, [&](int, long a, long b) {
        const long e = std::min<long>(n, b * 65536);
        for (long p = a * 65536; p < e; ++p)
            if (cell_i[p] < 1 || cell_i[p] > nii || cell_j[p] < 1 || cell_j[p] > njj) {
                int32_t o = bad.load();
                while (p < o && !bad.compare_exchange_weak(o, (int32_t)p)) {}
                break;
            }
    });
    return bad.load();
}

}  // namespace
