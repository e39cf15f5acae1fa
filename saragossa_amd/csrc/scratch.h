// Device scratch of a context's chunk calls, a buffer (and one for terms) per stream: launches on one stream are ordered by it,
// launches on different streams never share a buffer. Host bookkeeping only, over an interface of four device calls, so that
// tests/native/scratch.cpp runs it without a device.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <list>
#include <map>
#include <mutex>

namespace skv {

// What the scratch asks of the device; status 0 = done.
struct ScratchDevice {
    virtual int alloc(void **p, size_t bytes) = 0;
    virtual int free(void *p) = 0;
    virtual int wait_stream(void *stream) = 0;
    virtual int wait_device() = 0;
    virtual bool full(int status) = 0; // whether that status of alloc means that there is no memory

  protected:
    ~ScratchDevice() = default;
};

class StreamScratch {
    struct Buffer {
        void *ptr = nullptr;
        size_t bytes = 0;
        uint64_t used = 0; // value of clock_ at the last use
        int busy = 0;      // calls that are growing it or still queue launches that use it
        bool kept = false; // a captured launch has its address
    };

  public:
    // Buffers that no captured launch holds: a caller that makes a stream per request would otherwise leave one per dead
    // stream behind. Past that the least recently used one is dropped (after a wait for the device: its stream
    // may no longer exist).
    static constexpr size_t STREAMS = 8;
    static constexpr int REFUSED = -1; // a buffer would have to be replaced while its stream is being captured

    // From the moment a buffer is handed out until the call has queued the launches that use it: no other thread's call
    // drops it meanwhile.
    class Lease {
      public:
        Lease() = default;
        Lease(const Lease &) = delete;
        Lease &operator=(const Lease &) = delete;
        ~Lease() {
            if (!b_) return;
            std::lock_guard<std::mutex> lk(owner_->mu_);
            --b_->busy;
        }

      private:
        friend class StreamScratch;
        void take(StreamScratch *owner, Buffer *b) { // under the owner's lock
            if (b == b_) return;
            ++b->busy;
            if (b_) --b_->busy;
            owner_ = owner;
            b_ = b;
        }
        void drop() { // so, too
            if (b_) --b_->busy;
            b_ = nullptr;
        }
        StreamScratch *owner_ = nullptr;
        Buffer *b_ = nullptr;
    };

    // `need` bytes for launches on `stream`. Calls on one stream come from one thread at a time (as a stream's owner issues
    // its work anyway). A buffer handed out while its stream is being captured is in the graph for good: it is
    // never freed or replaced from then on while the scratch lives, a call that needs more gets one beside it, of twice its
    // size at least (so the buffers that stay are together no larger than the one in use). While a stream is being captured
    // nothing is waited for or freed, and a stream that has a buffer gets no larger one.
    // `optional`: the caller has a way with less. Nothing is given up for such a call: where there is no memory the stream
    // keeps the buffer it has, and as much is not asked for again before memory of the context has been freed.
    int get(ScratchDevice &dev, void *stream, size_t need, bool capturing, Lease &lease, void **out, bool optional = false) {
        *out = nullptr;
        {
            std::lock_guard<std::mutex> lk(mu_);
            auto it = streams_.find(stream);
            if (it != streams_.end() && it->second.bytes >= need) {
                Buffer &b = it->second;
                b.used = ++clock_;
                b.kept = b.kept || capturing;
                lease.take(this, &b);
                *out = b.ptr;
                return 0;
            }
            if (it != streams_.end() && it->second.ptr && capturing) return REFUSED;
            if (optional && need >= failed_) return REFUSED;
        }
        std::list<void *> aside(1, nullptr); // a node for what cannot be freed: to have it later takes no memory
        Buffer *b = nullptr;
        bool fresh = false;
        {
            std::lock_guard<std::mutex> lk(mu_);
            auto at = streams_.try_emplace(stream);
            b = &at.first->second;
            fresh = at.second;
            ++b->busy;
            if (fresh && !capturing) aside.front() = drop_oldest();
        }
        auto give_up = [&](int status) {
            std::lock_guard<std::mutex> lk(mu_);
            --b->busy;
            if (!b->ptr && b->busy == 0) streams_.erase(stream);
            return status;
        };
        auto keep_aside = [&]() {
            std::lock_guard<std::mutex> lk(mu_);
            kept_.splice(kept_.end(), aside);
        };
        // waits, frees and allocations outside the lock: calls on other streams go on meanwhile
        if (aside.front()) {
            int status = dev.wait_device();
            if (status != 0) {
                keep_aside();
                return give_up(status);
            }
            status = dev.free(aside.front());
            if (status != 0) return give_up(status);
        }
        void *p = nullptr;
        size_t bytes = b->kept ? std::max(need, 2 * b->bytes) : need;
        int status = dev.alloc(&p, bytes);
        if (status != 0 && bytes > need) {
            bytes = need;
            status = dev.alloc(&p, bytes);
        }
        if (status != 0 && optional) {
            if (dev.full(status)) {
                std::lock_guard<std::mutex> lk(mu_);
                failed_ = std::min(failed_, need);
            }
        } else if (status != 0 && b->ptr && !b->kept) { // in the place of the old one, which is of no use
            status = dev.wait_stream(stream); // work queued on the stream may still read it
            if (status == 0) {
                status = dev.free(b->ptr);
                std::lock_guard<std::mutex> lk(mu_);
                b->ptr = nullptr;
                b->bytes = 0;
            }
            if (status == 0) status = dev.alloc(&p, bytes);
        }
        if (status != 0) return give_up(status);
        void *old = b->ptr;
        const bool stays = b->kept;
        {
            std::lock_guard<std::mutex> lk(mu_);
            b->ptr = p;
            b->bytes = bytes;
            b->used = ++clock_;
            b->kept = capturing;
            lease.take(this, b);
            --b->busy;
        }
        if (old) {
            aside.front() = old;
            if (stays) keep_aside();
            else if ((status = dev.wait_stream(stream)) != 0) keep_aside();
            else status = dev.free(old);
            if (status != 0) return status;
        }
        *out = p;
        return 0;
    }

    // Room for the terms of f32 pages, a buffer of its own per stream, so that partials are never replaced for it: `want` bytes, or as
    // many as there are, `least` at least. Returns how many (at most `want`), 0 = none, and the caller takes its way without. The
    // buffers of all streams hold `limit` bytes at most. A buffer grows by a new one, the old one goes once that is there. Where
    // other streams' hold the room, those that the last IDLE calls did not use go. A size that there was no memory for is
    // not asked for again before memory of the context has been freed; half of it and a quarter are.
    static constexpr uint64_t IDLE = 64;
    size_t terms(ScratchDevice &dev, void *stream, size_t want, size_t least, size_t limit, Lease &lease, void **out) {
        *out = nullptr;
        {
            std::lock_guard<std::mutex> lk(mu_);
            auto it = terms_.find(stream);
            if (it != terms_.end() && it->second.bytes >= want) {
                it->second.used = ++clock_;
                lease.take(this, &it->second);
                *out = it->second.ptr;
                return want;
            }
        }
        std::list<void *> gone, old(1, nullptr);
        Buffer *b = nullptr;
        size_t ask = 0;
        {
            std::lock_guard<std::mutex> lk(mu_);
            b = &terms_.try_emplace(stream).first->second;
            lease.take(this, b);
            while (b->bytes < least && room(*b, limit) < least && drop_idle(gone)) {
            }
            ask = std::min(want, room(*b, limit));
        }
        if (!gone.empty()) give_back(dev, gone, dev.wait_device());
        void *p = nullptr;
        for (const size_t quarter = ask / 4; ask > b->bytes && ask >= least && ask >= quarter; ask /= 2) {
            {
                std::lock_guard<std::mutex> lk(mu_);
                if (ask >= failed_ || ask > room(*b, limit)) continue;
                terms_bytes_ += ask;
            }
            const int status = dev.alloc(&p, ask);
            if (status == 0) break;
            p = nullptr;
            std::lock_guard<std::mutex> lk(mu_);
            terms_bytes_ -= ask;
            if (!dev.full(status)) break;
            failed_ = std::min(failed_, ask);
        }
        {
            std::lock_guard<std::mutex> lk(mu_);
            if (p) {
                old.front() = b->ptr;
                terms_bytes_ -= b->bytes;
                b->ptr = p;
                b->bytes = ask;
            }
            if (b->bytes < least) {
                lease.drop();
                if (!b->ptr) terms_.erase(stream);
                return 0;
            }
            b->used = ++clock_;
            *out = b->ptr;
            ask = std::min(b->bytes, want);
        }
        if (old.front()) give_back(dev, old, dev.wait_stream(stream));
        return ask;
    }

    // Memory of the context has been freed: what there was none for may be asked for again.
    void freed() {
        std::lock_guard<std::mutex> lk(mu_);
        failed_ = SIZE_MAX;
    }

    // Everything; the caller has waited for the device and lets nobody use a buffer from here on.
    void drain(ScratchDevice &dev) {
        std::lock_guard<std::mutex> lk(mu_);
        for (auto *buffers : {&streams_, &terms_}) {
            for (auto &kv : *buffers)
                if (kv.second.ptr) (void)dev.free(kv.second.ptr);
            buffers->clear();
        }
        for (void *p : kept_) (void)dev.free(p);
        kept_.clear();
        terms_bytes_ = 0;
        failed_ = SIZE_MAX;
    }
    bool empty() {
        std::lock_guard<std::mutex> lk(mu_);
        return streams_.empty() && terms_.empty() && kept_.empty();
    }

  private:
    // Takes the least recently used buffer out where there are too many.
    void *drop_oldest() {
        size_t n = 0;
        auto oldest = streams_.end();
        for (auto it = streams_.begin(); it != streams_.end(); ++it) {
            if (!it->second.ptr || it->second.kept) continue;
            ++n;
            if (it->second.busy == 0 && (oldest == streams_.end() || it->second.used < oldest->second.used)) oldest = it;
        }
        if (n < STREAMS || oldest == streams_.end()) return nullptr;
        void *p = oldest->second.ptr;
        streams_.erase(oldest);
        return p;
    }

    // What the terms of a stream that has `own` may hold.
    size_t room(const Buffer &own, size_t limit) const {
        size_t n = 0;
        for (auto &kv : terms_) n += kv.second.ptr && &kv.second != &own;
        const size_t others = terms_bytes_ - own.bytes;
        return n >= STREAMS || others >= limit ? 0 : limit - others;
    }
    // Takes the terms out that were used longest ago, if no call uses them and IDLE calls have gone by.
    bool drop_idle(std::list<void *> &gone) {
        auto oldest = terms_.end();
        for (auto it = terms_.begin(); it != terms_.end(); ++it)
            if (it->second.ptr && it->second.busy == 0 && (oldest == terms_.end() || it->second.used < oldest->second.used)) oldest = it;
        if (oldest == terms_.end() || clock_ - oldest->second.used < IDLE) return false;
        gone.push_back(oldest->second.ptr);
        terms_bytes_ -= oldest->second.bytes;
        terms_.erase(oldest);
        failed_ = SIZE_MAX;
        return true;
    }
    // Frees buffers that have been waited for; those that could not be stay until the end.
    void give_back(ScratchDevice &dev, std::list<void *> &gone, int waited) {
        if (waited == 0) {
            for (void *p : gone) (void)dev.free(p);
            gone.clear();
        } else {
            std::lock_guard<std::mutex> lk(mu_);
            kept_.splice(kept_.end(), gone);
        }
    }

    std::mutex mu_;
    std::map<void *, Buffer> streams_;
    std::map<void *, Buffer> terms_;
    size_t terms_bytes_ = 0;    // of terms_, and what is being allocated for them
    size_t failed_ = SIZE_MAX;  // the least that there was no memory for
    std::list<void *> kept_; // of captured launches (or that could not be waited for), no longer a stream's own
    uint64_t clock_ = 0;
};

} // namespace skv
