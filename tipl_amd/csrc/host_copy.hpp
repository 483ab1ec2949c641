// host_copy.hpp -- the host side of a large device-to-host copy.  Plain C++
// (no HIP), so the logic also builds and is tested on a CPU-only host.
#pragma once

#include <condition_variable>
#include <cstddef>
#include <cstring>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace tiplhip {

// Copies `bytes` to `host` through a ring of `slots` staging chunks of
// `chunk` bytes.  issue(slot, offset, n) queues the transfer of n bytes from
// `offset` into the slot, arrived(slot) waits for it; both run on the calling
// thread, in order.  Up to `threads` threads, started for this copy and joined
// before it returns, move the chunks into place: what a copy into fresh
// memory costs is its page faults, and those run in parallel.  Where no
// thread can be started the calling one copies.  If issue or arrived throws,
// the threads are joined and the exception passes on (transfers may still be
// in flight into the slots: the caller drains them).
template <class Issue, class Arrived>
void staged_copy(char* host, size_t bytes, const char* staging, size_t chunk, size_t slots,
                 size_t threads, Issue&& issue, Arrived&& arrived)
{
    const size_t chunks = (bytes + chunk - 1) / chunk;
    auto size_of = [&](size_t c) { return c + 1 < chunks ? chunk : bytes - c * chunk; };
    std::mutex mu;
    std::condition_variable changed;
    size_t ready = 0, next = 0;      // chunks [0, ready) have arrived, [0, next) are taken
    std::vector<char> moved(chunks, 0);
    bool stop = false;
    auto work = [&] {
        std::unique_lock<std::mutex> lk(mu);
        for (;;) {
            changed.wait(lk, [&] { return stop || next < ready || next == chunks; });
            if (stop || next == chunks) return;
            const size_t c = next++;
            lk.unlock();
            std::memcpy(host + c * chunk, staging + (c % slots) * chunk, size_of(c));
            lk.lock();
            moved[c] = 1;
            changed.notify_all();
        }
    };
    struct Pool {
        std::vector<std::thread> t;
        std::mutex& mu;
        std::condition_variable& changed;
        bool& stop;
        bool finished = false;
        ~Pool()
        {
            if (!finished) {
                std::lock_guard<std::mutex> lk(mu);
                stop = true;
            }
            changed.notify_all();
            for (std::thread& x : t) x.join();
        }
    } pool{{}, mu, changed, stop};
    pool.t.reserve(threads);
    for (size_t i = 0; i < threads && i < chunks; ++i) {
        try {
            pool.t.emplace_back(work);
        } catch (const std::system_error&) {
            break;
        }
    }
    size_t issued = 0;
    for (size_t c = 0; c < chunks; ++c) {
        // transfers run ahead as far as the slots are free again
        for (; issued < chunks && issued < c + slots; ++issued) {
            if (issued >= slots) {
                std::unique_lock<std::mutex> lk(mu);
                if (!moved[issued - slots]) {
                    if (issued > c) break;
                    changed.wait(lk, [&] { return moved[issued - slots] != 0; });
                }
            }
            issue(issued % slots, issued * chunk, size_of(issued));
        }
        arrived(c % slots);
        if (pool.t.empty()) {
            std::memcpy(host + c * chunk, staging + (c % slots) * chunk, size_of(c));
            moved[c] = 1;
            continue;
        }
        {
            std::lock_guard<std::mutex> lk(mu);
            ready = c + 1;
        }
        changed.notify_all();
    }
    pool.finished = true;  // the threads leave when every chunk is taken
}

// Objects that several threads borrow, at most `limit` of them: take() lends an
// idle one, or one it makes while there are fewer, or none.  An object goes back
// when its lease ends; all are destroyed with the pool, which outlives them.
template <class T>
class BoundedPool {
public:
    explicit BoundedPool(size_t limit) : limit_(limit) {}
    BoundedPool(const BoundedPool&) = delete;
    BoundedPool& operator=(const BoundedPool&) = delete;

    class Lease {
    public:
        Lease() = default;
        Lease(BoundedPool* pool, std::unique_ptr<T> t) : pool_(pool), t_(std::move(t)) {}
        Lease(Lease&&) = default;
        Lease& operator=(Lease&&) = delete;
        ~Lease()
        {
            if (t_) pool_->put(std::move(t_));
        }
        explicit operator bool() const { return t_ != nullptr; }
        T* operator->() const { return t_.get(); }

    private:
        BoundedPool* pool_ = nullptr;
        std::unique_ptr<T> t_;
    };

    // make() returns a unique_ptr<T>; where it throws, the place stays free.
    template <class Make>
    Lease take(Make&& make)
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            if (!idle_.empty()) {
                std::unique_ptr<T> t = std::move(idle_.back());
                idle_.pop_back();
                return Lease(this, std::move(t));
            }
            if (made_ == limit_) return Lease();
            idle_.reserve(made_ + 1);  // put() never allocates
            ++made_;
        }
        try {
            return Lease(this, make());
        } catch (...) {
            std::lock_guard<std::mutex> lk(mu_);
            --made_;
            throw;
        }
    }

private:
    void put(std::unique_ptr<T> t)
    {
        std::lock_guard<std::mutex> lk(mu_);
        idle_.push_back(std::move(t));
    }

    const size_t limit_;
    std::mutex mu_;
    std::vector<std::unique_ptr<T>> idle_;
    size_t made_ = 0;
};

}  // namespace tiplhip
