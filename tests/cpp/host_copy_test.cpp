// staged_copy over sizes, ring depths and thread counts, against the source,
// and its behaviour when a transfer fails; BoundedPool's bound, from several
// threads, and its behaviour when an object cannot be made.
#include "../../tipl_amd/csrc/host_copy.hpp"

#include <atomic>
#include <cstdint>
#include <cstdio>
#include <stdexcept>

namespace {

int run(size_t bytes, size_t chunk, size_t slots, size_t threads)
{
    std::vector<char> src(bytes), dst(bytes, 0), staging(chunk * slots);
    for (size_t i = 0; i < bytes; ++i) src[i] = char(i * 2654435761u >> 13);
    std::vector<int> in_flight(slots, 0);
    tiplhip::staged_copy(
        dst.data(), bytes, staging.data(), chunk, slots, threads,
        [&](size_t s, size_t at, size_t n) {
            std::memcpy(&staging[s * chunk], &src[at], n);
            ++in_flight[s];
        },
        [&](size_t s) { --in_flight[s]; });
    for (int f : in_flight)
        if (f != 0) return 1;
    return std::memcmp(src.data(), dst.data(), bytes) != 0;
}

// At most `limit` objects at a time, each with one borrower, all destroyed with
// the pool.
int pool(size_t limit, int threads)
{
    static std::atomic<int> alive{0};
    struct Obj {
        std::atomic<int> users{0};
        Obj() { ++alive; }
        ~Obj() { --alive; }
    };
    std::atomic<int> bad{0}, lent{0}, none{0};
    {
        tiplhip::BoundedPool<Obj> p(limit);
        try {
            (void)p.take([]() -> std::unique_ptr<Obj> { throw std::bad_alloc(); });
            return 1;
        } catch (const std::bad_alloc&) {
        }
        std::vector<std::thread> t;
        for (int i = 0; i < threads; ++i)
            t.emplace_back([&] {
                for (int k = 0; k < 2000; ++k) {
                    auto l = p.take([] { return std::make_unique<Obj>(); });
                    if (!l) {
                        ++none;
                        continue;
                    }
                    ++lent;
                    if (++l->users != 1 || alive > int(limit)) ++bad;
                    --l->users;
                }
            });
        for (std::thread& x : t) x.join();
        std::vector<tiplhip::BoundedPool<Obj>::Lease> all;
        for (size_t i = 0; i < limit; ++i) all.push_back(p.take([] { return std::make_unique<Obj>(); }));
        for (auto& l : all)
            if (!l) ++bad;
        if (p.take([] { return std::make_unique<Obj>(); })) ++bad;
    }
    return bad != 0 || alive != 0 || lent == 0 || lent + none != threads * 2000;
}

}  // namespace

int main()
{
    for (size_t bytes : {1u, 63u, 64u, 65u, 640u, 1000u, 4096u, 100000u})
        for (size_t slots : {1u, 2u, 5u})
            for (size_t threads : {0u, 1u, 3u, 8u})
                if (run(bytes, 64, slots, threads)) {
                    std::printf("bytes %zu slots %zu threads %zu differ\n", bytes, slots, threads);
                    return 1;
                }
    std::vector<char> dst(1000), staging(128);
    bool thrown = false;
    try {
        tiplhip::staged_copy(
            dst.data(), dst.size(), staging.data(), 64, 2, 4, [&](size_t, size_t, size_t) {},
            [&](size_t) { throw std::runtime_error("transfer"); });
    } catch (const std::runtime_error&) {
        thrown = true;
    }
    if (!thrown) return 1;
    for (size_t limit : {1u, 4u})
        if (pool(limit, 8)) {
            std::printf("pool of %zu\n", limit);
            return 1;
        }
    std::printf("host copy ok\n");
    return 0;
}
