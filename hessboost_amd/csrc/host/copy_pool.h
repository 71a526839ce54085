// Large host copies shared among a few threads.
#pragma once
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>

namespace hbr {

// One thread's memcpy reaches a fraction of a host link's rate. The helpers
// are started once and serve every calling thread: a team of the compiler's
// parallel loops belongs to the thread that runs them, and each new thread's
// first copy waited 15 ms for its own. A copy is cut into pieces that the
// caller and whichever helpers are awake take in turn, so it never waits for
// a helper to wake (nor for any, in a forked child, which has none). One
// copy at a time.
class CopyPool {
public:
    explicit CopyPool(unsigned helpers) : s_(std::make_shared<State>()) {
        try {
            for (unsigned i = 0; i < helpers; i++) std::thread(help, s_).detach();
        } catch (const std::system_error &) {  // fewer helpers
        }
    }
    // The helpers end by themselves: they hold the state they share.
    ~CopyPool() {
        {
            std::lock_guard<std::mutex> lock(s_->mu);
            s_->stop = true;
        }
        s_->wake.notify_all();
    }
    CopyPool(const CopyPool &) = delete;
    CopyPool &operator=(const CopyPool &) = delete;

    void copy(void *dst, const void *src, uint64_t bytes) {
        if (bytes <= kPiece) {
            if (bytes) std::memcpy(dst, src, bytes);
            return;
        }
        const Job job{static_cast<char *>(dst), static_cast<const char *>(src), bytes};
        {
            std::lock_guard<std::mutex> lock(s_->mu);
            s_->job = job;
            s_->next = 0;
            s_->turn++;
        }
        s_->wake.notify_all();
        s_->take(job);
        // every piece is taken; those of the helpers still at work end soon
        // (a helper that comes now finds none, and leaves under the lock)
        std::unique_lock<std::mutex> lock(s_->mu);
        s_->idle.wait(lock, [&] { return s_->active == 0; });
        s_->job = Job{};
    }

private:
    static constexpr uint64_t kPiece = 256ull << 10;
    static constexpr int kSpin = 200;  // us
    struct Job {
        char *dst = nullptr;
        const char *src = nullptr;
        uint64_t bytes = 0;
    };
    struct State {
        std::mutex mu;
        std::condition_variable wake, idle;
        Job job;
        std::atomic<uint64_t> turn{0};
        unsigned active = 0;
        bool stop = false;
        std::atomic<uint64_t> next{0};
        void take(const Job &j) {
            for (;;) {
                const uint64_t at = next.fetch_add(1) * kPiece;
                if (at >= j.bytes) return;
                std::memcpy(j.dst + at, j.src + at, j.bytes - at < kPiece ? j.bytes - at : kPiece);
            }
        }
    };
    static void help(std::shared_ptr<State> s) {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> lock(s->mu);
        for (;;) {
            s->wake.wait(lock, [&] { return s->stop || s->turn != seen; });
            if (s->stop) return;
            seen = s->turn;
            const Job job = s->job;
            if (!job.bytes) continue;  // over already
            s->active++;
            lock.unlock();
            s->take(job);
            lock.lock();
            if (--s->active == 0) s->idle.notify_one();
            // the next chunk of the same call comes soon, and waking takes long
            lock.unlock();
            for (const auto end = std::chrono::steady_clock::now() + std::chrono::microseconds(kSpin);
                 s->turn == seen && std::chrono::steady_clock::now() < end;)
                std::this_thread::yield();
            lock.lock();
        }
    }
    std::shared_ptr<State> s_;
};

}  // namespace hbr
