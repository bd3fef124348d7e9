// fh3_fragments.h -- the device memory in which the large products' weights
// stand decoded (k_gemm256), shared by all calls.
//
// Rt stands for the HIP runtime, so that the rules below also run without a GPU:
//   Rt::Stream, Rt::Event (value types; Event{} is none)
//   bool capturing(Stream)          void *alloc(size_t)         void free(void *)
//   bool create(Event &)            bool wait(Stream, Event)    bool record(Event, Stream)
//   void sync(Event)                void destroy(Event)
#ifndef FH3_FRAGMENTS_H
#define FH3_FRAGMENTS_H

#include <stddef.h>

template <class Rt>
class WeightFragments {
public:
    using Stream = typename Rt::Stream;

    explicit WeightFragments(Rt r = Rt()) : rt(r) {}

    // Memory for one product on `st`; give() after its launches.  One buffer serves
    // every stream: each user waits on the device for the one before it.  NULL
    // -- the product then reads its weights in place (k_gemm, the same bits) --
    // when the stream is being captured (a graph must not hold the shared
    // buffer or wait for events outside it) or the memory is not to be had.
    void *take(size_t bytes, Stream st) {
        if (rt.capturing(st)) return nullptr;
        if (cap < bytes) {
            if (!grow(bytes)) return nullptr;
        } else if (!rt.wait(st, used)) {
            return nullptr;
        }
        return p;
    }

    // The product's launches are on `st`; false: the caller must wait for them.
    bool give(Stream st) { return rt.record(used, st); }

    void clear() {
        if (p) rt.free(p);
        if (used != typename Rt::Event{}) rt.destroy(used);
        p = nullptr, cap = 0, used = {};
    }

private:
    // The old buffer stays until the new one is there, and for good if it is refused.
    bool grow(size_t bytes) {
        if (used == typename Rt::Event{} && !rt.create(used)) return false;
        void *q = rt.alloc(bytes);
        if (!q) return false;
        if (p) {
            rt.sync(used);
            rt.free(p);
        }
        p = q, cap = bytes;
        return true;
    }

    Rt rt;
    void *p = nullptr;
    size_t cap = 0;
    typename Rt::Event used{};  // after the last product that read p
};

#endif
