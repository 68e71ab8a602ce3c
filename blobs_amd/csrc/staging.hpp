// staging.hpp -- pinned memory through which exports bring state to the host
// (World::export_state), and the events of its two halves.
//
// An allocation costs some 200 us, as much as ten reads of a small world, so a
// buffer is lent for one read at a time and goes back to a pool that outlives
// worlds: it grows with the reads that run at once, one per thread.  Idle
// buffers are at most kIdle; when the last world ends, all but the small ones
// are freed.  Every call may come from any thread.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <vector>

namespace bg {

class Staging {
public:
    // Halves are of at least kLeast and at most kHalf bytes.
    static constexpr size_t kLeast = 32 << 10, kHalf = 4 << 20;

    Staging() = default;
    ~Staging() {
        if (b_.mem) pool().give_back(b_);
    }
    Staging(const Staging&) = delete;
    Staging& operator=(const Staging&) = delete;

    // A buffer whose halves hold `bytes` (or kHalf, if that is less).  `device` is the current
    // one, and nothing on it uses the buffer when this ends.
    hipError_t take(size_t bytes, int device) { return pool().take(bytes, device, b_); }
    char* half(uint32_t i) const { return b_.mem + i * b_.half; }
    size_t half_bytes() const { return b_.half; }
    hipEvent_t event(uint32_t i) const { return b_.event[i]; }

    // Worlds alive, counted by their constructors and destructors.
    static void world_begins() { pool().worlds(1); }
    static void world_ends() { pool().worlds(-1); }

private:
    struct Buffer {
        int device = -1;
        char* mem = nullptr;  // two halves
        size_t half = 0;
        hipEvent_t event[2] = {nullptr, nullptr};
    };
    static void release(Buffer& b) {
        if (b.mem) (void)hipHostFree(b.mem);
        for (hipEvent_t e : b.event)
            if (e) (void)hipEventDestroy(e);
        b = Buffer{};
    }
    class Pool {
    public:
        hipError_t take(size_t bytes, int device, Buffer& out) {
            const size_t half = std::min(kHalf, std::max((bytes + 4095) & ~(size_t)4095, kLeast));
            {
                std::lock_guard<std::mutex> lock(mu_);
                size_t best = idle_.size();
                for (size_t i = 0; i < idle_.size(); ++i)
                    if (idle_[i].device == device && idle_[i].half >= half &&
                        (best == idle_.size() || idle_[i].half < idle_[best].half))
                        best = i;
                if (best < idle_.size()) {
                    out = idle_[best];
                    idle_.erase(idle_.begin() + (std::ptrdiff_t)best);
                    return hipSuccess;
                }
            }
            Buffer b;
            b.device = device;
            b.half = half;
            hipError_t e = hipHostMalloc((void**)&b.mem, 2 * half, hipHostMallocDefault);
            for (hipEvent_t& ev : b.event)
                if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
            if (e != hipSuccess) release(b);
            out = b;
            return e;
        }
        void give_back(Buffer& b) {
            Buffer drop;
            {
                std::lock_guard<std::mutex> lock(mu_);
                idle_.push_back(b);
                b = Buffer{};
                if (idle_.size() > kIdle) {  // the one idle for longest
                    drop = idle_.front();
                    idle_.erase(idle_.begin());
                }
            }
            release(drop);
        }
        void worlds(int by) {
            std::vector<Buffer> drop;
            {
                std::lock_guard<std::mutex> lock(mu_);
                worlds_ += by;
                if (worlds_ > 0) return;
                for (size_t i = idle_.size(); i-- > 0;)
                    if (idle_[i].half > kSmall) {
                        drop.push_back(idle_[i]);
                        idle_.erase(idle_.begin() + (std::ptrdiff_t)i);
                    }
            }
            for (Buffer& b : drop) release(b);
        }

    private:
        static constexpr size_t kIdle = 4, kSmall = 256 << 10;
        std::mutex mu_;
        std::vector<Buffer> idle_;
        long worlds_ = 0;
    };
    static Pool& pool() {
        static Pool* p = new Pool;  // (never destroyed: the HIP runtime may be gone by then)
        return *p;
    }
    Buffer b_;
};

}  // namespace bg
