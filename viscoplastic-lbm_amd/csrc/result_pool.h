// Result buffers of a batch's jobs. Released ones are kept for later jobs, at
// most kKeptBytes of them in a batch: a fresh buffer costs its page faults, as much
// time as its copy. One thread may release results while another advances the
// batch, so the pool has a lock.
#pragma once
#include <cstddef>
#include <map>
#include <memory>
#include <mutex>
#include <new>
#include <utility>

namespace vlbm {
namespace detail {

class ResultPool {
public:
    static constexpr size_t kKeptBytes = size_t(256) << 20;

    // A buffer of at least `bytes`, its size in *got; null when the host has no memory.
    std::unique_ptr<char[]> take(size_t bytes, size_t* got) {
        {
            std::lock_guard<std::mutex> lock(mu_);
            auto best = spare_.lower_bound(bytes);
            if (best != spare_.end() && best->first <= 2 * bytes) {
                *got = best->first;
                std::unique_ptr<char[]> p = std::move(best->second);
                kept_ -= best->first;
                spare_.erase(best);
                return p;
            }
        }
        *got = bytes;
        return std::unique_ptr<char[]>(new (std::nothrow) char[bytes]);
    }
    void give(std::unique_ptr<char[]> p, size_t bytes) {
        std::lock_guard<std::mutex> lock(mu_);
        if (!p || kept_ + bytes > kKeptBytes) return;
        try {
            spare_.emplace(bytes, std::move(p));
            kept_ += bytes;
        } catch (const std::bad_alloc&) {               // then it is freed
        }
    }

private:
    std::mutex mu_;
    std::multimap<size_t, std::unique_ptr<char[]>> spare_;
    size_t kept_ = 0;
};

}  // namespace detail
}  // namespace vlbm
