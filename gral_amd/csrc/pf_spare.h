// Device memory that its owner can do without: the strips' buffers of a tall
// situation, which runs per-diagonal (the same results, slower) without them.  An
// allocation that fails anywhere else in the process takes it back, so such
// situations keep no other out of memory.
//
// The owner holds Spare::use during every call that uses the memory and asks keep(),
// once it has it, whether the memory is still there.  SparePool::give_back frees the
// memory of one spare that is not in use; with wait, and if all are in use, it waits
// for the end of one's call (the owner's next call then gives the memory back by
// itself, whichever of the two comes first).  A thread that waits must hold no
// spare's lock.  A spare without memory is in no pool.  Plain host code; release
// frees one pointer.
#pragma once
#include <algorithm>
#include <atomic>
#include <memory>
#include <mutex>
#include <vector>

struct Spare {
    std::mutex use;
    std::vector<void *> mem;               // empty: given back (guarded by use)
    std::atomic<bool> wanted{false};
    int device = -1;
    void (*release)(void *) = nullptr;
    void free_all() {                      // with use held
        for (void *p : mem) release(p);
        mem.clear();
    }
};

class SparePool {
    std::mutex mu_;
    std::vector<std::shared_ptr<Spare>> all_;

public:
    void add(const std::shared_ptr<Spare> &s) {
        std::lock_guard<std::mutex> g(mu_);
        all_.push_back(s);
    }
    void remove(const std::shared_ptr<Spare> &s) {
        std::lock_guard<std::mutex> g(mu_);
        all_.erase(std::remove(all_.begin(), all_.end(), s), all_.end());
    }
    // frees the memory of one spare of the device other than own (or finds that its
    // owner just did); false: there is none left, or without wait none idle
    bool give_back(int device, const Spare *own, bool wait) {
        std::vector<std::shared_ptr<Spare>> now;
        {
            std::lock_guard<std::mutex> g(mu_);
            for (auto &s : all_)
                if (s.get() != own && s->device == device) now.push_back(s);
        }
        for (auto &s : now) {
            std::unique_lock<std::mutex> l(s->use, std::try_to_lock);
            if (!l.owns_lock()) continue;
            s->free_all();
            remove(s);
            return true;
        }
        if (!wait || now.empty()) return false;
        auto &s = now.front();
        s->wanted.store(true);
        std::lock_guard<std::mutex> l(s->use);
        s->free_all();
        remove(s);
        return true;
    }
    // with use held, by the owner at the start of a call: whether the memory is still
    // there; gives it back if another thread waits for it
    bool keep(const std::shared_ptr<Spare> &s) {
        if (s->wanted.load() && !s->mem.empty()) {
            s->free_all();
            remove(s);
        }
        return !s->mem.empty();
    }
};
