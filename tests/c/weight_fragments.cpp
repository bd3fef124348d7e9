// The rules of fh3_fragments.h against a runtime that only keeps books: every
// step prints nothing and returns its line on failure.
#include <cstdio>
#include <map>
#include <set>
#include <vector>

#include "fh3_fragments.h"

struct Books {
    size_t limit = 1u << 30, held = 0;  // bytes the "device" has, and how many are allocated
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
    bool capturing(int st) { return b.captured.count(st) != 0; }
    void *alloc(size_t n) {
        b.allocs++;
        if (b.held + n > b.limit) return nullptr;
        void *p = ::operator new(1);
        b.live[p] = n;
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
    void sync(int e) { b.busy.erase(e); }
};

#define CHECK(x) \
    if (!(x)) return std::printf("line %d: %s\n", __LINE__, #x), __LINE__

static int growth() {
    b = Books();
    b.limit = 500;
    WeightFragments<Fake> w;
    void *p = w.take(100, 1);
    CHECK(p && w.give(1));
    CHECK(!w.take(450, 1));                        // both do not fit: refused ...
    CHECK(b.live.count(p) && w.take(100, 1) == p);  // ... and the one that was there still serves
    w.give(1);
    void *q = w.take(300, 1);
    CHECK(q && q != p && b.held == 300);  // the old one goes once the new one is there
    w.give(1);
    CHECK(w.take(100, 1) == q);
    w.give(1);
    w.clear();
    CHECK(b.held == 0);
    return 0;
}

static int capture() {
    b = Books();
    WeightFragments<Fake> w;
    b.captured.insert(7);
    CHECK(!w.take(100, 7) && b.allocs == 0);
    return 0;
}

int main() {
    if (int r = growth()) return r;
    if (int r = capture()) return r;
    return 0;
}
