// The upload ring's bookkeeping against a GPU that reads nothing until it is
// waited for: no byte is handed out again while an upload that used it may
// still be unread. Arguments: seed, then the upload sizes to choose from. Exit
// status 1 on the first byte handed out too early.
#include "half_ring.hpp"

#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

int main(int argc, char** argv) {
    constexpr std::size_t kHalf = std::size_t(1) << 20;
    struct Upload {
        std::size_t begin, end;
    };
    std::mt19937 rng(unsigned(std::atoi(argv[1])));
    std::vector<std::size_t> sizes;
    for (int i = 2; i < argc; ++i) sizes.push_back(std::size_t(std::atoll(argv[i])));

    vchip::HalfRing ring(kHalf);
    std::vector<Upload> uploads;                  // in stream order
    std::size_t done = 0, marked[2] = {0, 0};     // uploads read for certain; uploads before each half's last mark
    std::size_t waits = 0;
    for (int k = 0; k < 20000; ++k) {
        const std::size_t n = (sizes[rng() % sizes.size()] + 15) / 16 * 16;
        const std::size_t at = ring.take(
            n, [&](int half) { marked[half] = uploads.size(); },
            [&](int half) {
                ++waits;
                if (marked[half] > done) done = marked[half];
            });
        if (at + n > 2 * kHalf || (at < kHalf && at + n > kHalf)) {
            std::printf("upload %d: bytes %zu to %zu leave their half\n", k, at, at + n);
            return 1;
        }
        for (std::size_t i = done; i < uploads.size(); ++i)
            if (uploads[i].begin < at + n && at < uploads[i].end) {
                std::printf("upload %d takes bytes %zu to %zu while upload %zu may be unread\n", k, at, at + n, i);
                return 1;
            }
        uploads.push_back({at, at + n});
    }
    std::printf("%zu waits\n", waits);
    return 0;
}
