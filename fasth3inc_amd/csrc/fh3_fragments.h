// fh3_fragments.h -- the device memory in which the large products' weights
// stand decoded (k_gemm256), shared by all calls.
//
// Rt stands for the HIP runtime, so that the rules below also run without a GPU:
//   Rt::Stream, Rt::Event (value types; Event{} is none)
//   bool capturing(Stream)          void *alloc(size_t)         void free(void *)
//   size_t available()  (bytes of device memory that are free)
//   Rt::On(int)  (the device is the calling thread's current one while it lives)
//   bool create(Event &)            bool wait(Stream, Event)    bool record(Event, Stream)
//   bool done(Event)                void sync(Event)            void destroy(Event)
#ifndef FH3_FRAGMENTS_H
#define FH3_FRAGMENTS_H

#include <stddef.h>

template <class Rt>
class WeightFragments {
public:
    using Stream = typename Rt::Stream;

    explicit WeightFragments(Rt r = Rt()) : rt(r) {}

    // Memory for one product on `st`; give() after its launches.  A stream has
    // its own buffer, up to SLOTS of them, so that products on different streams
    // run side by side; a further stream takes one whose work has ended.  NULL -- the
    // product then reads its weights in place (k_gemm, the same bits) -- when
    // all are at work for others, when the stream is being captured (a graph must
    // not hold a shared buffer or wait for events outside it) or the memory is
    // not to be had.  No stream ever waits for another.
    // (2048 x 5120 -> 5120 on two streams: 124 us a product with one buffer whose
    // users waited for one another, 102 with k_gemm alone, 98 with two.)
    // Memory and events are the library's device's, whichever the calling thread's is.
    void *take(size_t bytes, Stream st, int device) {
        if (rt.capturing(st)) return nullptr;
        Slot *s = pick(bytes, st);
        if (!s) return nullptr;
        if (s->cap < bytes) {
            typename Rt::On here(device);
            if (!grow(*s, bytes)) return nullptr;
        } else if (!rt.wait(st, s->used)) {  // for earlier work of this stream, or of one whose handle it has
            return nullptr;
        }
        s->last = st;
        taken = s;
        return s->p;
    }

    // The product's launches are on `st`; false: the caller must wait for them.
    bool give(Stream st) { return rt.record(taken->used, st); }

    // Every buffer back to the device, once its work has ended; false: there was none.
    bool trim() {
        bool any = false;
        for (Slot &s : slots)
            if (s.p) {
                rt.sync(s.used);
                rt.free(s.p);
                s.p = nullptr, s.cap = 0;
                any = true;
            }
        return any;
    }

    void clear() {
        for (Slot &s : slots) {
            if (s.p) rt.free(s.p);
            if (s.used != Event{}) rt.destroy(s.used);
            s = Slot();
        }
    }

private:
    using Event = typename Rt::Event;
    struct Slot {
        void *p = nullptr;
        size_t cap = 0;
        Event used{};   // after the last product that read p
        Stream last{};  // its stream
    };
    static constexpr int SLOTS = 2;

    // Large enough and this stream's, or idle; else to be grown: this
    // stream's, an unused one, an idle one.
    Slot *pick(size_t bytes, Stream st) {
        Slot *own = nullptr, *unused = nullptr, *idle = nullptr, *fit = nullptr;
        for (Slot &s : slots) {
            if (!s.p) {
                if (!unused) unused = &s;
                continue;
            }
            const bool mine = s.last == st;
            if (!mine && !rt.done(s.used)) continue;
            if (s.cap >= bytes && (!fit || mine)) fit = &s;
            (mine ? own : idle) = &s;
        }
        return fit ? fit : own ? own : unused ? unused : idle;
    }

    // The old buffer stays until the new one is there, and for good if it is refused.
    // At most an eighth of the free memory is taken: k_gemm needs none, and what is
    // left is the caller's.
    bool grow(Slot &s, size_t bytes) {
        if (bytes > rt.available() / 8) return false;
        if (s.used == Event{} && !rt.create(s.used)) return false;
        void *q = rt.alloc(bytes);
        if (!q) return false;
        if (s.p) {
            rt.sync(s.used);
            rt.free(s.p);
        }
        s.p = q, s.cap = bytes;
        return true;
    }

    Rt rt;
    Slot slots[SLOTS], *taken = nullptr;
};

#endif
