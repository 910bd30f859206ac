// Threads that take and release result buffers at once: a program that collects
// results in one thread while another advances the batch.
#include <atomic>
#include <cstdio>
#include <cstring>
#include <thread>
#include <vector>

#include "result_pool.h"

int main() {
    vlbm::detail::ResultPool pool;
    std::atomic<int> wrong{0};
    std::vector<std::thread> threads;
    for (int t = 0; t < 8; t++)
        threads.emplace_back([&, t] {
            for (int r = 0; r < 20000; r++) {
                const size_t bytes = 64 + (size_t)(r * 37 + t * 101) % 1000;
                size_t got = 0;
                auto p = pool.take(bytes, &got);
                if (!p || got < bytes || got > 2 * bytes) { wrong++; continue; }
                std::memset(p.get(), t, got);
                std::this_thread::yield();
                for (size_t k = 0; k < got; k += 61)
                    if (p[k] != (char)t) wrong++;                    // somebody else holds it too
                pool.give(std::move(p), got);
            }
        });
    for (auto& t : threads) t.join();
    std::printf("%d wrong\n", wrong.load());
    return wrong ? 1 : 0;
}
