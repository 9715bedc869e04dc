// mg_hostpack.hpp -- the threads that pack a caller's host arrays into pinned
// buffers, or unpack them (host_fields): host code only.
#pragma once
#include <array>
#include <atomic>
#include <exception>
#include <thread>

namespace mf3d {

// copy(f, q) copies piece q of field f to or from the buffer of field f; the
// threads take the pieces in order, field by field, and wait at a field that
// is not open yet.  Field f is open once open(n), n > f, was called: its buffer
// may be used.  wait(f) returns when every piece of field f is copied.
//
// Starting a thread fails where the process may have no more of them or no more
// memory: the ones that run then do all the work, and the caller
// does it where start() returns 0.  Nothing here throws, and no thread
// outlives the object: the destructor ends those that wait and joins all.
template <typename Copy>
class PackTeam {
public:
    static constexpr int kThreads = 8, kFields = 8;

    PackTeam(int fields, int pieces, const Copy &copy) : nf_(fields), np_(pieces), copy_(copy) {
        for (auto &c : copied_) c = 0;
    }
    PackTeam(const PackTeam &) = delete;
    PackTeam &operator=(const PackTeam &) = delete;
    ~PackTeam() {
        stop_ = true;
        for (int t = 0; t < running_; ++t) threads_[t].join();
    }

    // Up to `want` threads; how many run.
    int start(int want) noexcept {
        try {
            while (running_ < want && running_ < kThreads) {
                threads_[running_] = std::thread([this] { work(); });
                ++running_;
            }
        } catch (const std::exception &) {  // std::system_error, std::bad_alloc
        }
        return running_;
    }
    void open(int fields) { open_.store(fields, std::memory_order_release); }
    void wait(int f) const {
        while (copied_[f].load(std::memory_order_acquire) < np_) std::this_thread::yield();
    }

private:
    void work() {
        for (;;) {
            const int c = next_.fetch_add(1);
            if (c >= nf_ * np_) return;
            const int f = c / np_;
            while (open_.load(std::memory_order_acquire) <= f) {
                if (stop_.load()) return;
                std::this_thread::yield();
            }
            copy_(f, c % np_);
            copied_[f].fetch_add(1, std::memory_order_release);
        }
    }

    const int nf_, np_;
    const Copy &copy_;
    std::atomic<int> next_{0}, open_{0};
    std::atomic<bool> stop_{false};
    std::array<std::atomic<int>, kFields> copied_;
    std::array<std::thread, kThreads> threads_;
    int running_ = 0;
};

}  // namespace mf3d
