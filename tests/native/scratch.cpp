// The bookkeeping of a context's device scratch (saragossa_amd/csrc/scratch.h) over a device that only counts: what
// a captured launch holds stays, nothing is waited for or freed during a capture, nothing leaks or is freed
// twice, whatever fails.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>
#include <set>
#include <vector>

#include "scratch.h"

using skv::StreamScratch;

#define CHECK(cond)                                                        \
    do {                                                                   \
        if (!(cond)) {                                                     \
            std::printf("FAIL line %d: %s\n", __LINE__, #cond);            \
            std::exit(1);                                                  \
        }                                                                  \
    } while (0)

struct Device final : skv::ScratchDevice {
    std::map<void *, size_t> live;
    size_t held = 0, room = SIZE_MAX;
    int allocs = 0, frees = 0, waits = 0, failing_waits = 0;
    char *next = reinterpret_cast<char *>(0x10000);
    int alloc(void **p, size_t bytes) override {
        ++allocs;
        if (bytes > room - held) return 2;
        *p = next;
        next += bytes + 256;
        live[*p] = bytes;
        held += bytes;
        return 0;
    }
    int free(void *p) override {
        ++frees;
        CHECK(live.count(p) == 1);
        held -= live[p];
        live.erase(p);
        return 0;
    }
    int wait_stream(void *) override { return wait_device(); }
    int wait_device() override {
        ++waits;
        return failing_waits > 0 ? (--failing_waits, 3) : 0;
    }
    bool full(int status) override { return status == 2; }
    int calls() const { return allocs + frees + waits; }
};

static void *stream(int i) { return reinterpret_cast<void *>((uintptr_t)i * 64); }

static void *got(StreamScratch &s, Device &d, int i, size_t need, bool capturing = false) {
    StreamScratch::Lease lease;
    void *p = nullptr;
    CHECK(s.get(d, stream(i), need, capturing, lease, &p) == 0 && d.live.at(p) >= need);
    return p;
}

static int refusal(StreamScratch &s, Device &d, int i, size_t need, bool capturing = false) {
    StreamScratch::Lease lease;
    void *p = nullptr;
    const int status = s.get(d, stream(i), need, capturing, lease, &p);
    CHECK(status != 0 && !p);
    return status;
}

static void captured_buffers_stay() {
    Device d;
    StreamScratch s;
    void *first = got(s, d, 1, 1000);
    CHECK(got(s, d, 1, 800) == first && d.allocs == 1);
    CHECK(got(s, d, 1, 900, true) == first); // a graph has it now
    void *second = got(s, d, 1, 1100);       // an eager call of more
    CHECK(second != first && d.live.count(first) && d.live.at(second) >= 2000 && d.frees == 0);
    void *third = got(s, d, 1, 5000);        // nobody captured the second one
    CHECK(d.live.count(first) && !d.live.count(second) && d.live.count(third));
    CHECK(got(s, d, 1, 10) == third);
    // too small while the stream is being captured: refused before anything is done
    const int before = d.calls();
    CHECK(refusal(s, d, 1, 6000, true) == StreamScratch::REFUSED);
    CHECK(d.calls() == before && got(s, d, 1, 5000, true) == third);
    // a stream that has none may allocate (where the capture lets it), but waits for and frees nothing
    for (int i = 2; i < 20; ++i) got(s, d, i, 100);
    const int waits = d.waits, frees = d.frees;
    void *other = got(s, d, 30, 64, true);
    CHECK(d.waits == waits && d.frees == frees);
    d.room = d.held;
    CHECK(refusal(s, d, 31, 64, true) == 2);
    CHECK(d.waits == waits && d.frees == frees);
    d.room = SIZE_MAX;
    // nor does another stream's call drop what a graph has, however long ago that was
    for (int i = 40; i < 80; ++i) got(s, d, i, 100);
    CHECK(d.live.count(first) && d.live.count(third) && d.live.count(other));
    CHECK(d.live.size() == 3 + StreamScratch::STREAMS);
    s.drain(d);
    CHECK(d.live.empty() && s.empty());
}

static void oldest_goes() {
    Device d;
    StreamScratch s;
    std::vector<void *> p;
    for (int i = 0; i < 8; ++i) p.push_back(got(s, d, i, 100));
    got(s, d, 0, 100); // used again: stream 1's is the oldest now
    {
        StreamScratch::Lease lease; // a call of stream 1 that has its buffer and has not queued its launches yet
        void *q = nullptr;
        CHECK(s.get(d, stream(1), 100, false, lease, &q) == 0 && q == p[1]);
        for (int i = 8; i < 40; ++i) got(s, d, i, 100);
        CHECK(d.live.count(p[1]) && !d.live.count(p[0]));
    }
    got(s, d, 41, 100);
    CHECK(!d.live.count(p[1]) && d.live.size() == 8);
    s.drain(d);
    CHECK(d.live.empty());
}

static void failures() {
    Device d;
    StreamScratch s;
    void *small = got(s, d, 1, 600);
    d.room = 1000; // no room for both: the old one goes first
    void *large = got(s, d, 1, 900);
    CHECK(!d.live.count(small) && d.live.count(large) && d.waits == 1);
    CHECK(refusal(s, d, 1, 2000) == 2 && d.live.empty() && s.empty()); // nothing helps
    d.room = SIZE_MAX;
    void *old = got(s, d, 1, 100);
    d.failing_waits = 1;
    CHECK(refusal(s, d, 1, 200) == 3 && d.live.count(old)); // not waited for: not freed
    got(s, d, 1, 200);
    s.drain(d);
    CHECK(d.live.empty() && s.empty());
    for (int i = 0; i < 8; ++i) got(s, d, i, 100);
    d.failing_waits = 1;
    CHECK(refusal(s, d, 9, 100) == 3 && d.live.size() == 8);
    got(s, d, 9, 100);
    s.drain(d);
    CHECK(d.live.empty() && s.empty());
}

static void random_calls() {
    std::mt19937 rng(5);
    for (int run = 0; run < 200; ++run) {
        Device d;
        StreamScratch s;
        std::set<void *> captured;
        for (int call = 0; call < 300; ++call) {
            const int i = (int)(rng() % 24);
            const size_t need = 1 + rng() % 5000;
            const bool capturing = rng() % 6 == 0;
            d.room = rng() % 10 == 0 ? d.held + rng() % 2000 : SIZE_MAX;
            d.failing_waits = rng() % 20 == 0 ? 1 : 0;
            const int waits = d.waits, frees = d.frees;
            StreamScratch::Lease lease;
            void *p = nullptr;
            const int status = s.get(d, stream(i), need, capturing, lease, &p);
            if (capturing) CHECK(d.waits == waits && d.frees == frees);
            CHECK((status == 0) == (p != nullptr));
            if (p) CHECK(d.live.at(p) >= need);
            if (p && capturing) captured.insert(p);
            for (void *c : captured) CHECK(d.live.count(c));
        }
        s.drain(d);
        CHECK(d.live.empty() && s.empty());
    }
}

static size_t terms(StreamScratch &s, Device &d, int i, size_t want, size_t least, size_t limit, void **out = nullptr) {
    StreamScratch::Lease lease;
    void *p = nullptr;
    const size_t n = s.terms(d, stream(i), want, least, limit, lease, &p);
    CHECK(n <= want && (n == 0) == (p == nullptr) && (n == 0 || (n >= least && d.live.at(p) >= n)));
    if (out) *out = p;
    return n;
}

static void terms_beside_partials() {
    Device d;
    StreamScratch s;
    void *partials = got(s, d, 1, 1000), *a = nullptr, *b = nullptr;
    CHECK(terms(s, d, 1, 500, 100, 10000, &a) == 500 && a != partials);
    CHECK(terms(s, d, 1, 300, 300, 10000, &b) == 300 && b == a);
    CHECK(terms(s, d, 1, 5000, 600, 10000, &b) == 5000 && !d.live.count(a) && d.live.count(partials));
    CHECK(got(s, d, 1, 1000) == partials); // never replaced for terms
    // no memory: what there is serves, nothing is freed or waited for, and the size is asked for once
    d.room = d.held + 100;
    const int frees = d.frees, waits = d.waits;
    CHECK(terms(s, d, 1, 9000, 600, 10000) == 5000);
    int allocs = d.allocs;
    CHECK(terms(s, d, 1, 9000, 600, 10000) == 5000 && d.allocs == allocs);
    CHECK(terms(s, d, 1, 9500, 5500, 10000) == 0 && d.allocs == allocs);
    CHECK(terms(s, d, 2, 4000, 4000, 10000) == 0);
    allocs = d.allocs;
    CHECK(terms(s, d, 2, 4000, 4000, 10000) == 0 && d.allocs == allocs);
    StreamScratch::Lease lease;
    void *p = nullptr;
    CHECK(s.get(d, stream(1), 4100, false, lease, &p, true) != 0 && d.allocs == allocs); // optional partials: not tried either
    CHECK(s.get(d, stream(1), 1500, false, lease, &p, true) != 0 && d.allocs == allocs + 1);
    CHECK(s.get(d, stream(1), 1500, false, lease, &p, true) != 0 && d.allocs == allocs + 1);
    CHECK(got(s, d, 1, 1000) == partials && d.frees == frees && d.waits == waits);
    s.freed();
    d.room = SIZE_MAX;
    CHECK(terms(s, d, 1, 9000, 600, 10000) == 9000 && d.live.size() == 2);
    CHECK(terms(s, d, 1, 700, 600, 10000, &a) == 700);
    // half of what is wanted, or a quarter, where there is that
    d.room = d.held + 450;
    CHECK(terms(s, d, 3, 1000, 100, 20000, &b) == 500 / 2);
    CHECK(d.live.at(b) == 250);
    d.room = SIZE_MAX;
    CHECK(terms(s, d, 3, 1000, 100, 20000) == 250); // still remembered
    s.freed();
    CHECK(terms(s, d, 3, 1000, 100, 20000) == 1000 && !d.live.count(b));
}

static void terms_of_many_streams() {
    Device d;
    StreamScratch s;
    void *first = nullptr, *p = nullptr;
    CHECK(terms(s, d, 1, 600, 100, 1000, &first) == 600);
    CHECK(terms(s, d, 2, 600, 100, 1000) == 400); // what is left
    CHECK(terms(s, d, 3, 600, 100, 1000) == 0 && d.held == 1000);
    for (int i = 0; i < 100; ++i) CHECK(terms(s, d, 2, 600, 100, 1000) == 400); // (stream 1 is idle)
    CHECK(terms(s, d, 3, 600, 100, 1000) == 600 && !d.live.count(first) && d.held == 1000);
    {
        StreamScratch::Lease lease; // a call of stream 3 that still queues launches
        CHECK(s.terms(d, stream(3), 600, 100, 1000, lease, &p) == 600);
        for (int i = 0; i < 100; ++i) CHECK(terms(s, d, 2, 400, 100, 1000) == 400);
        CHECK(terms(s, d, 4, 600, 100, 1000) == 0 && d.live.count(p));
    }
    for (int i = 0; i < 100; ++i) CHECK(terms(s, d, 2, 400, 100, 1000) == 400);
    CHECK(terms(s, d, 4, 600, 100, 1000) == 600 && !d.live.count(p));
    CHECK(terms(s, d, 2, 300, 1, 0) == 300); // a lower limit takes nothing away
    CHECK(terms(s, d, 2, 500, 450, 0) == 0);
    for (int i = 10; i < 40; ++i) terms(s, d, i, 1, 1, 100000);
    CHECK(d.live.size() == StreamScratch::STREAMS);
    d.failing_waits = 1;
    CHECK(terms(s, d, 2, 50000, 1, 100000) == 50000 && d.live.size() == StreamScratch::STREAMS + 1);
    s.drain(d);
    CHECK(d.live.empty() && s.empty());
    std::mt19937 rng(9);
    for (int call = 0; call < 20000; ++call) {
        const size_t want = 1 + rng() % 3000;
        d.room = rng() % 4 == 0 ? d.held + rng() % 2000 : SIZE_MAX;
        if (rng() % 100 == 0) s.freed();
        if (rng() % 3 == 0) d.room = SIZE_MAX, (void)got(s, d, (int)(rng() % 12), 1 + rng() % 100);
        terms(s, d, (int)(rng() % 12), want, 1 + want / 8, 6000);
    }
    s.drain(d);
    CHECK(d.live.empty() && s.empty());
}

int main() {
    captured_buffers_stay();
    oldest_goes();
    failures();
    random_calls();
    terms_beside_partials();
    terms_of_many_streams();
    std::puts("ok");
    return 0;
}
