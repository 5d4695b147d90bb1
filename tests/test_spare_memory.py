"""The strips' buffers of tall situations make room for every other allocation (pf_spare.h).

Host code, compiled and run here on a stand-in for the device's memory: situations of
12 units each that take 19 more where they find them fill a memory of 12 N units with
N of them; a spare in use is left alone, or awaited; an owner that starts call after call
gives way to a thread that waits; another device's are not touched."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gral_amd", "csrc")
SOURCE = r"""
#include <cassert>
#include <chrono>
#include <cstdint>
#include <cstdio>
#include <thread>
#include "pf_spare.h"
#undef NDEBUG
#include <cassert>
static std::atomic<int> room{0};
static void release(void *p) { room += (int)(intptr_t)p; }
static bool take(int n) {
    for (int r = room; r >= n;)
        if (room.compare_exchange_weak(r, r - n)) return true;
    return false;
}
static std::shared_ptr<Spare> spare(SparePool &pool, int n, int device) {
    auto s = std::make_shared<Spare>();
    s->release = release;
    s->device = device;
    s->mem = {(void *)(intptr_t)n};
    pool.add(s);
    return s;
}
int main() {
    {
        SparePool pool;
        std::vector<std::shared_ptr<Spare>> held;
        const int N = 40;
        room = 12 * N;
        for (int q = 0; q < N; ++q) {
            while (!take(12)) assert(pool.give_back(0, nullptr, true));
            if (take(19)) held.push_back(spare(pool, 19, 0));
        }
        assert(room >= 0 && room < 12 && held.size() == 12 * N / 31);
        for (auto &s : held) assert(!pool.keep(s));       // all of them are back
        assert(!pool.give_back(0, nullptr, true));
    }
    {
        SparePool pool;
        room = 0;
        auto a = spare(pool, 5, 0), b = spare(pool, 7, 1);
        assert(!pool.give_back(0, a.get(), true));        // its own, another device's
        {
            std::lock_guard<std::mutex> l(a->use);
            assert(pool.keep(a));
            std::thread t([&] { assert(!pool.give_back(0, nullptr, false)); });       // in use
            t.join();
        }
        assert(room == 0);
        std::atomic<bool> in{false}, stop{false}, gone{false};
        std::thread owner([&] {                           // call after call
            while (!stop) {
                std::lock_guard<std::mutex> l(a->use);
                in = true;
                if (!pool.keep(a)) gone = true;
                else std::this_thread::sleep_for(std::chrono::milliseconds(2));
            }
        });
        while (!in) std::this_thread::yield();
        assert(pool.give_back(0, nullptr, true));
        assert(room == 5);
        while (!gone) std::this_thread::yield();
        stop = true;
        owner.join();
        assert(pool.give_back(1, nullptr, false) && room == 12 && !pool.give_back(1, nullptr, true));
    }
    {
        SparePool pool;                                   // removed by its owner while another waits
        room = 0;
        auto a = spare(pool, 5, 0);
        a->use.lock();
        std::thread t([&] { assert(pool.give_back(0, nullptr, true)); });
        while (!a->wanted) std::this_thread::yield();
        a->free_all();
        pool.remove(a);
        a->use.unlock();
        t.join();
        assert(room == 5 && !pool.give_back(0, nullptr, true));
    }
    std::puts("ok");
}
"""


def test_spare_pool(tmp_path):
    src, exe = tmp_path / "s.cpp", tmp_path / "s"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True, timeout=60).stdout == "ok\n"
