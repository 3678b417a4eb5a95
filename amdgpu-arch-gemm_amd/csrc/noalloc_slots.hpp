// Which part of sgemm_launch_noalloc's scratch a call works in, and what it
// waits for first.  Host only; no HIP: `Streams` is the stream runtime, so that
// the rules run against a model of it in a test.
//
// The scratch is cut into kSlots slots, each owned by the stream whose calls
// used it last.  A call that fits a slot takes its stream's own one, a free one,
// or the one longest unused; a larger call takes them all.  Work of another
// owner is waited for on the device, by an event recorded on its stream when the
// slot is taken over: a call on a slot that its stream owns costs nothing.
//
// A stream that is capturing can neither be recorded on (the event would join
// its graph) nor be assumed idle (eager calls from before its capture may still
// run), so its slots cannot be taken over: a call that needs one gets kBusy and
// runs without scratch.
//
// Captured calls run when their graph is replayed, which is the caller's to
// order against everything else on the device: they leave the owners alone.
// Those of one capture all begin at the first slot and become a chain of
// dependent nodes, also where its streams branch.
//
// A name that stands for another stream in every thread (hipStreamPerThread)
// cannot be recorded on later from elsewhere: its calls record the slot's own
// event at once, which every later call on the slot waits for.
#pragma once

#include <cstddef>
#include <cstdint>

namespace noalloc {

constexpr int kSlots = 8;
constexpr int kBusy = -1000;   // no scratch for this call now

// Streams:
//   typedef ... Stream;
//   bool capturing(Stream s, uint64_t* id)   whether s is capturing, in which capture
//   bool per_thread(Stream s)                whether the name means another stream in every thread
//   uint64_t thread()                        the calling thread
//   int order(Stream before, Stream after)   later work of `after` waits for the work enqueued on `before`;
//                                            kBusy: `before` began a capture meanwhile, nothing waits
//   int mark(int slot, Stream s)             the slot's event: the work enqueued on s so far
//   int wait(int slot, Stream s)             later work of s waits for the slot's event
//   int sync(Stream s)                       waits for s on the host
// and every int is 0 on success.
template <class Streams> class Slots {
  public:
    typedef typename Streams::Stream Stream;

    // Takes one slot (all: every slot) for the call that is enqueued on `s`
    // next.  *first: its slot; *fresh: its tickets may be another stream's;
    // *captured: the call is part of a capture.
    int take(Streams& streams, Stream s, bool all, int* first, bool* fresh, bool* captured) {
        uint64_t id = 0;
        *first = 0;
        *fresh = *captured = streams.capturing(s, &id);
        if (*captured) return take_captured(streams, s, id);
        const bool named = streams.per_thread(s);
        auto own = [&](const Slot& t) { return t.state == kOwned && t.owner == s && !named; };
        if (!all)
            for (Slot& t : slots_)
                if (own(t)) {
                    *first = (int)(&t - slots_);
                    t.used = ++calls_;
                    return 0;
                }
        uint64_t other = 0;
        bool stuck[kSlots];
        for (int q = 0; q < kSlots; ++q)
            stuck[q] = slots_[q].state == kOwned && !own(slots_[q]) && streams.capturing(slots_[q].owner, &other);
        if (!all) {
            auto rank = [&](int q) { return slots_[q].state == kFree ? 1 : !stuck[q] ? 2 : 3; };
            for (int q = 1; q < kSlots; ++q)
                if (rank(q) < rank(*first) || (rank(q) == rank(*first) && slots_[q].used < slots_[*first].used)) *first = q;
        }
        const int end = all ? kSlots : *first + 1;
        for (int q = *first; q < end; ++q)
            if (stuck[q]) return kBusy;
        for (int q = *first; q < end; ++q) {
            Slot& t = slots_[q];
            if (!own(t)) {
                *fresh = true;
                bool waited = t.state == kFree;
                for (int p = *first; p < q && !waited; ++p) waited = t.state == kOwned && was_[p] && old_[p] == t.owner;
                if (!waited) {
                    const int e = t.state == kMarked ? streams.wait(q, s) : streams.order(t.owner, s);
                    if (e) return e;
                }
            }
            was_[q] = t.state == kOwned;
            old_[q] = t.owner;
        }
        for (int q = *first; q < end; ++q) {
            slots_[q].state = kOwned;
            slots_[q].owner = s;
            slots_[q].used = calls_ + 1;
        }
        ++calls_;
        return 0;
    }

    // After the call's launch on `s` (same lock as its take).
    int done(Streams& streams, Stream s, bool all, int first) {
        uint64_t id = 0;
        if (!streams.per_thread(s) || streams.capturing(s, &id)) return 0;
        for (int q = first; q < (all ? kSlots : first + 1); ++q) {
            const int e = streams.mark(q, s);
            if (e) return e;
            slots_[q].state = kMarked;
        }
        return 0;
    }

    // `s` is about to be destroyed, or a handle leaves it: its slots are free
    // once its work has ended (calls of other handles on it included, which the
    // lock keeps out meanwhile).
    int forget(Streams& streams, Stream s) {
        bool any = false;
        for (const Slot& t : slots_) any = any || (t.state == kOwned && t.owner == s);
        for (Chain& c : chains_)
            if (c.last == s) c.on = false;
        if (!any) return 0;
        const int e = streams.sync(s);
        for (Slot& t : slots_)
            if (t.state == kOwned && t.owner == s) t.state = kFree;
        return e;
    }

  private:
    enum State { kFree, kOwned, kMarked };
    struct Slot {
        State state = kFree;
        Stream owner = Stream();
        uint64_t used = 0;
    };
    // The captured calls of one capture: the stream (and thread, for a
    // per-thread name) of the last one.
    struct Chain {
        bool on = false;
        uint64_t id = 0, thread = 0;
        Stream last = Stream();
    };
    Slot slots_[kSlots];
    bool was_[kSlots];
    Stream old_[kSlots];
    uint64_t calls_ = 0;
    Chain chains_[kSlots];   // captures at once; one more runs without scratch

    int take_captured(Streams& streams, Stream s, uint64_t id) {
        const uint64_t thread = streams.per_thread(s) ? streams.thread() : 0;
        Chain* mine = nullptr;
        Chain* unused = nullptr;
        for (Chain& c : chains_) {
            if (c.on && c.id == id) mine = &c;
            uint64_t other = 0;
            const bool elsewhere = c.thread && c.thread != streams.thread();   // cannot be asked from here
            if (!c.on || (!elsewhere && c.id != id && !(streams.capturing(c.last, &other) && other == c.id))) unused = &c;
        }
        if (mine && !(mine->last == s && mine->thread == thread)) {
            if (mine->thread && mine->thread != streams.thread()) return kBusy;
            const int e = streams.order(mine->last, s);
            if (e) return e;
        }
        if (!mine) mine = unused;
        if (!mine) return kBusy;
        mine->on = true;
        mine->id = id;
        mine->last = s;
        mine->thread = thread;
        return 0;
    }
};

}  // namespace noalloc
