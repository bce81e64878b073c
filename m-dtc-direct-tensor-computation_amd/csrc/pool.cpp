// pool.cpp -- idle device and page-locked memory kept from one call or object for the next
// (dtc_internal.hpp states who may put what in, and the bounds).
#include <chrono>
#include <iterator>
#include <list>
#include <map>
#include <mutex>

#include "dtc_internal.hpp"

namespace dtc {

thread_local bool t_recycle = false;

namespace {

struct Pool {
    using Clock = std::chrono::steady_clock;
    struct Block {
        void* p;
        size_t n;
        int dev;
        Clock::time_point since;
    };
    std::mutex mu;
    std::list<Block> idle;                                                         // newest first
    std::multimap<std::pair<int, size_t>, std::list<Block>::iterator> by_size;
    size_t bytes = 0;
    std::list<Block> pinned;                                                       // page-locked words, newest first

    // unlinks the oldest blocks while over the bound or past their time; the caller frees them
    void expire(std::list<Block>& out, size_t bound) {
        const Clock::time_point now = Clock::now();
        while (!idle.empty() &&
               (bytes > bound || std::chrono::duration<double>(now - idle.back().since).count() > POOL_SECONDS)) {
            const auto last = std::prev(idle.end());
            auto r = by_size.equal_range({last->dev, last->n});
            while (r.first->second != last) ++r.first;
            by_size.erase(r.first);
            bytes -= last->n;
            out.splice(out.begin(), idle, last);
        }
    }

    // the same for the page-locked words
    void expire_pinned(std::list<Block>& out, size_t bound) {
        const Clock::time_point now = Clock::now();
        while (!pinned.empty() && (pinned.size() > bound ||
                                   std::chrono::duration<double>(now - pinned.back().since).count() > POOL_SECONDS))
            out.splice(out.begin(), pinned, std::prev(pinned.end()));
    }
};

// never destroyed: the runtime may be gone when static objects are
Pool& pool() {
    static Pool& p = *new Pool;
    return p;
}

void free_blocks(const std::list<Pool::Block>& v) {
    for (const Pool::Block& b : v) (void)hipFree(b.p);
}

void free_words(const std::list<Pool::Block>& v) {
    for (const Pool::Block& b : v) (void)hipHostFree(b.p);
}

}  // namespace

void* pool_take(size_t n, int dev) {
    Pool& P = pool();
    void* p = nullptr;
    std::list<Pool::Block> old;
    {
        std::lock_guard<std::mutex> lk(P.mu);
        const auto it = P.by_size.find({dev, n});
        if (it != P.by_size.end()) {
            p = it->second->p;
            P.bytes -= n;
            P.idle.erase(it->second);
            P.by_size.erase(it);
        }
        P.expire(old, POOL_BYTES);
    }
    free_blocks(old);
    return p;
}

void pool_put(void* p, size_t n, int dev) {
    Pool& P = pool();
    std::list<Pool::Block> old;
    {
        std::lock_guard<std::mutex> lk(P.mu);
        // (called from destructors: without host memory for the entry the block is freed; so is
        // one that would push most of the others out)
        std::list<Pool::Block> one;
        if (n <= POOL_BYTES / 4) try {
            one.push_front({p, n, dev, Pool::Clock::now()});
            P.by_size.emplace(std::make_pair(dev, n), one.begin());
            P.idle.splice(P.idle.begin(), one);
            P.bytes += n;
            p = nullptr;
        } catch (...) {
        }
        P.expire(old, POOL_BYTES);
    }
    if (p) (void)hipFree(p);
    free_blocks(old);
}

void pool_trim() {
    Pool& P = pool();
    std::list<Pool::Block> old, words;
    {
        std::lock_guard<std::mutex> lk(P.mu);
        P.expire(old, 0);
        words.swap(P.pinned);
    }
    free_blocks(old);
    free_words(words);
}

void* pool_take_pinned(size_t n) {
    Pool& P = pool();
    void* p = nullptr;
    std::list<Pool::Block> old;
    {
        std::lock_guard<std::mutex> lk(P.mu);
        for (auto it = P.pinned.begin(); it != P.pinned.end(); ++it)
            if (it->n == n) {
                p = it->p;
                P.pinned.erase(it);
                break;
            }
        P.expire_pinned(old, POOL_PINNED);
    }
    free_words(old);
    return p;
}

void pool_put_pinned(void* p, size_t n) {
    Pool& P = pool();
    std::list<Pool::Block> old;
    {
        std::lock_guard<std::mutex> lk(P.mu);
        std::list<Pool::Block> one;
        if (n <= POOL_PINNED_BYTES) try {
            one.push_front({p, n, 0, Pool::Clock::now()});
            P.pinned.splice(P.pinned.begin(), one);
            p = nullptr;
        } catch (...) {
        }
        P.expire_pinned(old, POOL_PINNED);
    }
    if (p) (void)hipHostFree(p);
    free_words(old);
}

}  // namespace dtc

extern "C" int dtc_release_memory(void) {
    dtc::pool_trim();
    return DTC_OK;
}
