// staged_copy over sizes, ring depths and thread counts, against the source;
// and its behaviour when a transfer fails.
#include "../../tipl_amd/csrc/host_copy.hpp"

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
    std::printf("host copy ok\n");
    return 0;
}
