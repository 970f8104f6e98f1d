// ff_launch_order.hpp -- the bookkeeping behind WaitingLaunch (ff_runtime.hpp)
// for one device. Host only and without GPU calls.
#pragma once

namespace ffamd {

struct LaunchOrder {
    unsigned target = 0;          // awaited tiles of the launches enqueued so far (modulo 2^32)
    const void* last = nullptr;   // stream of the last of them (the null stream is a stream too)
    bool pending = false;         // it may not have started

    bool marked = false;          // an event was recorded on its stream right before it
    int marks = 0;                // launches that are still to be marked

    // What a launch on s has to wait for first.
    //  GATE: the last launch was marked. The event and then a kernel that polls
    //        the count of starts up to target: whatever the last launch's
    //        stream had queued before it is waited for by the event, however
    //        long that takes, and the poll spans its own start only.
    //  END:  it was not. An event after it, or the device.
    // (The launches before the last need no look: the last one waited for them.)
    enum class Before { NOTHING, GATE, END };
    Before before(const void* s) const {
        if (!pending || last == s) return Before::NOTHING;
        return marked ? Before::GATE : Before::END;
    }
    // Launches are marked only while streams take turns before their work is
    // done: an event between two frames of one stream costs some microseconds.
    // kMarks after the last such switch they stop, and the next one waits for
    // the last launch's end.
    static constexpr int kMarks = 64;
    void switched() { marks = kMarks; }
    bool mark() const { return marks > 0; }
    // A launch on s whose tiles will count `awaited` starts was enqueued, with
    // or without a mark. Only what really was enqueued is noted: a failed
    // launch starts nothing, and a start that is expected but never comes would
    // hold up every later switch of streams, one that comes unexpected would
    // let them through too early.
    void launched(const void* s, int awaited, bool with_mark) {
        target += (unsigned)awaited;
        last = s;
        pending = true;
        marked = with_mark;
        if (marks > 0) --marks;
    }
    // All that was enqueued on s is done.
    void finished(const void* s) {
        if (last == s) pending = false;
    }
    // All that was enqueued on the device is done, and the count stands at n.
    void restart(unsigned n) {
        target = n;
        pending = false;
    }
};

}  // namespace ffamd
