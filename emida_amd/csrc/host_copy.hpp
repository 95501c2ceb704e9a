// Copies from pageable host memory, shared by the host entry points.
//
// One core copies a pattern at about 28 GB/s out of DRAM (1.5 MB: 53 us), half of what the
// link to the GPU takes; the runtime's own pageable upload of it takes 86 us.  copy_team
// splits a copy into chunks that the calling thread and a few helper threads claim in order,
// so the first part can be on its way while the rest is copied.  One host call (873 x 873
// uint16, 400 ROIs): 129 -> 90 us; 64 requests of such patterns to a server, whose submissions
// were bound by this copy: 4.5 -> 2.7 ms.
#pragma once
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace emida_amd {

class copy_team {
  public:
    // Below this a copy is not worth waking anybody (256 KB: 9 us on one core).
    static constexpr size_t kMin = 512 << 10;

    // The process's team while anybody holds it; its threads end with the last holder.
    static std::shared_ptr<copy_team> get() {
        static std::mutex mu;
        static std::weak_ptr<copy_team> current;
        std::lock_guard<std::mutex> lock(mu);
        auto p = current.lock();
        if (!p) current = p = std::make_shared<copy_team>();
        return p;
    }

    copy_team() {
        cpu_set_t set;
        const int cpus = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
        const int n = std::min(kHelpers, cpus / 4);
        helpers.reserve(n > 0 ? n : 0);  // from here on only the threads themselves can fail
        try {
            for (int i = 0; i < n; ++i) helpers.emplace_back([this] { work(); });
        } catch (const std::system_error&) {  // fewer helpers, or none
        }
    }
    ~copy_team() {
        {
            std::lock_guard<std::mutex> lock(mu);
            stop = true;
            gen.fetch_add(1);
        }
        cv.notify_all();
        for (auto& t : helpers) t.join();
    }
    copy_team(const copy_team&) = delete;

    // Copies n bytes.  ready(m), called by this thread as the first m bytes have been copied,
    // m growing, the last time n; it must not throw.  One copy at a time has the helpers, one
    // that finds them taken copies alone.
    template <class F>
    void copy(void* dst, const void* src, size_t n, F&& ready) {
        std::unique_lock<std::mutex> owner(busy, std::defer_lock);
        if (helpers.empty() || n < kMin || !owner.try_lock()) {
            std::memcpy(dst, src, n);
            ready(n);
            return;
        }
        {
            std::lock_guard<std::mutex> lock(mu);
            j.dst = (char*)dst;
            j.src = (const char*)src;
            j.n = n;
            j.chunk = std::max(kChunk, (n / kMaxChunks + 4096) & ~(size_t)4095);
            j.count = (uint32_t)((n + j.chunk - 1) / j.chunk);
            for (uint32_t i = 0; i < j.count; ++i) j.done[i].store(false, std::memory_order_relaxed);
            j.next.store(0, std::memory_order_relaxed);
            open = true;
            gen.fetch_add(1);
        }
        cv.notify_all();
        uint32_t prefix = 0;
        auto tell = [&] {
            const uint32_t before = prefix;
            while (prefix < j.count && j.done[prefix].load(std::memory_order_acquire)) ++prefix;
            if (prefix > before) ready(std::min(n, prefix * j.chunk));
        };
        while (step()) tell();
        while (prefix < j.count) {
            pause();
            tell();
        }
        {
            std::lock_guard<std::mutex> lock(mu);
            open = false;
        }
        while (active.load(std::memory_order_acquire)) pause();  // helpers past their last chunk
    }
    void copy(void* dst, const void* src, size_t n) {
        copy(dst, src, n, [](size_t) {});
    }

  private:
    static constexpr int kHelpers = 3;
    static constexpr size_t kChunk = 64 << 10;
    static constexpr size_t kMaxChunks = 256;

    static void pause() {
#if defined(__x86_64__)
        __builtin_ia32_pause();
#else
        std::this_thread::yield();
#endif
    }
    // Claims and copies one chunk; false when there is none left.
    bool step() {
        const uint32_t i = j.next.fetch_add(1, std::memory_order_relaxed);
        if (i >= j.count) return false;
        const size_t at = i * j.chunk;
        std::memcpy(j.dst + at, j.src + at, std::min(j.chunk, j.n - at));
        j.done[i].store(true, std::memory_order_release);
        return true;
    }
    void work() {
        uint32_t seen = 0;
        while (true) {
            // copies often come in a row (a request after the other): look for about 30 us
            // before sleeping, waking takes longer than a chunk
            for (int i = 0; i < 600 && gen.load(std::memory_order_acquire) == seen; ++i) pause();
            {
                std::unique_lock<std::mutex> lock(mu);
                cv.wait(lock, [&] { return gen.load() != seen; });
                seen = gen.load();
                if (stop) return;
                if (!open) continue;
                active.fetch_add(1);
            }
            while (step()) {
            }
            active.fetch_sub(1, std::memory_order_release);
        }
    }

    struct job {
        char* dst = nullptr;
        const char* src = nullptr;
        size_t n = 0, chunk = 0;
        uint32_t count = 0;
        std::atomic<uint32_t> next{0};
        std::atomic<bool> done[kMaxChunks];
    };
    std::mutex busy;  // held by the copy that has the helpers
    std::mutex mu;    // job, open, stop; helpers join a copy under it
    std::condition_variable cv;
    job j;
    bool open = false, stop = false;
    std::atomic<uint32_t> gen{0};
    std::atomic<int> active{0};  // helpers inside the current copy
    std::vector<std::thread> helpers;
};

}  // namespace emida_amd
