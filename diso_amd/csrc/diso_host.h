// diso_host.h - host-side helpers of the waiting forward: how a thread waits for a word that a kernel
// writes, and objects that host threads take turns to own.
//
// Plain C++, so both are testable on the CPU.
#pragma once

#include <stdint.h>
#include <time.h>

#include <mutex>
#include <vector>

namespace diso_host {

inline int64_t now_ns() {
    timespec t;
    clock_gettime(CLOCK_MONOTONIC, &t);
    return (int64_t)t.tv_sec * 1000000000 + t.tv_nsec;
}

// Waits until done() or until trouble() (looked at now and then) gives a nonzero code, which is
// returned. Polls for the first millisecond, which covers a count (tens to hundreds of microseconds)
// and some work ahead of it; a longer wait sleeps a sixteenth of the time waited so far between looks
// (at most a millisecond), so that it costs neither a core nor more than that sixteenth.
constexpr int64_t kPollNs = 1000000, kMaxSleepNs = 1000000;
template <class Done, class Trouble>
inline int wait_until(Done done, Trouble trouble) {
    const int64_t start = now_ns();
    for (uint32_t looks = 1;; ++looks) {
        if (done()) return 0;
        if (looks % 1024 != 0) {
            __builtin_ia32_pause();
            continue;
        }
        const int64_t waited = now_ns() - start;
        if (waited >= kPollNs || looks % 4096 == 0) {
            const int rc = trouble();
            if (rc) return rc;
        }
        if (waited >= kPollNs) {
            const int64_t ns = waited / 16 < kMaxSleepNs ? waited / 16 : kMaxSleepNs;
            const timespec t{0, ns};
            nanosleep(&t, nullptr);
            looks = 1023;  // one look, then here again
        }
    }
}

// An object per host thread, taken over by a later thread when its owner ends: as many are made as
// threads have held one at a time.
template <class T, T *(*Make)()>
T *thread_object() {
    struct Pool {
        std::mutex mu;
        std::vector<T *> free;
    };
    static Pool *const pool = new Pool;  // (outlives every thread)
    struct Holder {
        T *obj = nullptr;
        ~Holder() {
            if (!obj) return;
            std::lock_guard<std::mutex> lock(pool->mu);
            pool->free.push_back(obj);
        }
    };
    static thread_local Holder mine;
    if (!mine.obj) {
        {
            std::lock_guard<std::mutex> lock(pool->mu);
            if (!pool->free.empty()) {
                mine.obj = pool->free.back();
                pool->free.pop_back();
            }
        }
        if (!mine.obj) mine.obj = Make();
    }
    return mine.obj;
}

}  // namespace diso_host
