// The rules of fh3_fragments.h against a runtime that only keeps books: every
// step prints nothing and returns its line on failure.
#include <cstdio>
#include <map>
#include <set>
#include <vector>

#include "fh3_fragments.h"

struct Books {
    size_t limit = 1u << 30, held = 0;  // bytes the "device" has, and how many are allocated
    int device = 0;                     // the thread's current one
    std::map<void *, int> home;         // the device of each allocation
    size_t hidden = 0;                  // free bytes that no allocation gets
    int allocs = 0, events = 0;
    std::map<void *, size_t> live;
    std::set<int> busy;        // events whose work has not ended
    std::set<int> captured;    // streams under capture
    std::vector<int> waits;    // events waited for on the device
};
static Books b;

struct Fake {
    using Stream = int;
    using Event = int;
    struct On {
        int old = b.device;
        explicit On(int d) { b.device = d; }
        ~On() { b.device = old; }
    };
    bool capturing(int st) { return b.captured.count(st) != 0; }
    size_t available() { return b.limit - b.held; }
    void *alloc(size_t n) {
        b.allocs++;
        if (b.held + n > b.limit - b.hidden) return nullptr;
        void *p = ::operator new(1);
        b.live[p] = n;
        b.home[p] = b.device;
        b.held += n;
        return p;
    }
    void free(void *p) {
        b.held -= b.live.at(p);
        b.live.erase(p);
        ::operator delete(p);
    }
    bool create(int &e) { return (e = ++b.events) != 0; }
    void destroy(int) {}
    bool wait(int, int e) { return b.waits.push_back(e), true; }
    bool record(int e, int) { return b.busy.insert(e), true; }
    bool done(int e) { return !b.busy.count(e); }
    void sync(int e) { b.busy.erase(e); }
};

#define CHECK(x) \
    if (!(x)) return std::printf("line %d: %s\n", __LINE__, #x), __LINE__

static int growth() {
    b = Books();
    b.limit = 5000, b.hidden = 4500;
    WeightFragments<Fake> w;
    void *p = w.take(100, 1, 0);
    CHECK(p && w.give(1));
    CHECK(!w.take(450, 1, 0));                        // both do not fit: refused ...
    CHECK(b.live.count(p) && w.take(100, 1, 0) == p);  // ... and the one that was there still serves
    w.give(1);
    void *q = w.take(300, 1, 0);
    CHECK(q && q != p && b.held == 300);  // the old one goes once the new one is there
    w.give(1);
    CHECK(w.take(100, 1, 0) == q);
    w.give(1);
    w.clear();
    CHECK(b.held == 0);
    return 0;
}

static int capture() {
    b = Books();
    WeightFragments<Fake> w;
    b.captured.insert(7);
    CHECK(!w.take(100, 7, 0) && b.allocs == 0);
    return 0;
}

// Streams 1, 2 and 3 at work at once: two buffers, no stream waits for another
// and no buffer is used under one that is still at work.
static int streams() {
    b = Books();
    WeightFragments<Fake> w;
    void *p = w.take(100, 1, 0);
    CHECK(p && w.give(1));
    void *q = w.take(100, 2, 0);
    CHECK(q && q != p && w.give(2) && b.waits.empty());
    CHECK(!w.take(100, 3, 0) && !w.take(10, 3, 0) && b.waits.empty() && b.allocs == 2);
    CHECK(w.take(100, 1, 0) == p && w.give(1));  // behind its own stream's work
    CHECK(b.waits == std::vector<int>{1});
    CHECK(w.take(100, 2, 0) == q && w.give(2));
    b.busy.erase(1);  // stream 1's work ends: a third stream takes its buffer
    CHECK(w.take(100, 3, 0) == p && w.give(3));
    CHECK(!w.take(100, 1, 0) && b.allocs == 2);
    void *r = w.take(200, 2, 0);  // a stream's own buffer grows behind its work, the others stay
    CHECK(r && w.give(2) && b.live.count(p) && !b.live.count(q) && b.held == 300);
    b.busy.clear();
    CHECK(w.take(150, 3, 0) == r && w.give(3));  // the idle one is large enough: no growth
    CHECK(b.allocs == 3);
    w.clear();
    CHECK(b.held == 0);
    return 0;
}

// Memory that others need is left to them, and given back when they ask.
static int memory() {
    b = Books();
    b.limit = 1000;
    WeightFragments<Fake> w;
    CHECK(!w.take(126, 1, 0) && b.allocs == 0);  // more than an eighth of what is free
    CHECK(w.take(125, 1, 0) && w.give(1));
    CHECK(!w.take(110, 2, 0) && b.allocs == 1);  // of what is free now
    CHECK(w.take(109, 2, 0) && w.give(2) && b.held == 234);
    CHECK(w.trim() && b.held == 0 && b.busy.empty() && !w.trim());
    CHECK(w.take(125, 2, 0) && w.give(2));
    return 0;
}

// A thread whose current device is another one.
static int device() {
    b = Books();
    WeightFragments<Fake> w;
    void *p = w.take(100, 1, 3);
    CHECK(p && b.home.at(p) == 3 && b.device == 0);
    return 0;
}

int main() {
    if (int r = device()) return r;
    if (int r = memory()) return r;
    if (int r = streams()) return r;
    if (int r = growth()) return r;
    if (int r = capture()) return r;
    return 0;
}
