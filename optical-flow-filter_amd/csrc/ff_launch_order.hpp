// ff_launch_order.hpp -- the bookkeeping behind WaitingLaunch (ff_runtime.hpp)
// for one device. Host only and without GPU calls.
#pragma once

namespace ffamd {

struct LaunchOrder {
    unsigned target = 0;          // awaited tiles of the launches enqueued so far (modulo 2^32)
    const void* last = nullptr;   // stream of the last of them (the null stream is a stream too)
    bool pending = false;         // it may not have started

    // Whether a launch on s has to come after the last one.
    bool follows(const void* s) const { return pending && last != s; }
    // A launch on s whose tiles will count `awaited` starts was enqueued. Only
    // what really was enqueued is noted: a failed launch starts nothing, and a
    // start that is expected but never comes would hold up every later switch
    // of streams, one that comes unexpected would let them through too early.
    void launched(const void* s, int awaited) {
        target += (unsigned)awaited;
        last = s;
        pending = true;
    }
    // All that was enqueued on s is done.
    void finished(const void* s) {
        if (last == s) pending = false;
    }
};

}  // namespace ffamd
