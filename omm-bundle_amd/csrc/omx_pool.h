// Device memory of omx_malloc: freed blocks kept mapped for later allocations.
#pragma once

#include <hip/hip_runtime_api.h>

#include <map>
#include <mutex>
#include <vector>

namespace omx {

// hipFree unmaps (0.2 ms for a 34 MB matrix) and hipMalloc maps again (0.06 ms); an omm() call makes and
// frees 17 matrices, which for 1458 x 2916 was 4.4 of its 11.1 ms (6.8 without).  A freed block therefore stays mapped
// until an allocation of up to an eighth less asks for it, it is the oldest of too many (64 blocks, 1/64 of
// the device's memory: a block beyond that is freed at once), an allocation fails, or a context ends.  Shared by all contexts and threads: a block
// becomes idle only after a wait for the whole device, as in hipFree (device_wait), so whichever stream takes it
// next finds no work left on it, and omx_malloc clears it like a new one.
class DevPool {
  public:
    // An idle block of at least `bytes` on the current device, or null.
    void *take(size_t bytes) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return nullptr;
        std::lock_guard<std::mutex> lock(mu_);
        size_t best = idle_.size();
        for (size_t q = 0; q < idle_.size(); ++q)
            if (idle_[q].dev == dev && idle_[q].bytes >= bytes && idle_[q].bytes <= bytes + bytes / 8 &&
                (best == idle_.size() || idle_[q].bytes < idle_[best].bytes))
                best = q;
        if (best == idle_.size()) return nullptr;
        const Block b = idle_[best];
        live_[b.p] = b;  // may throw: the block is still idle then
        idle_.erase(idle_.begin() + best);
        held_ -= b.bytes;
        return b.p;
    }
    // Notes a new block of the current device; without the note it is freed as any other memory.
    void note(void *p, size_t bytes) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return;
        std::lock_guard<std::mutex> lock(mu_);
        live_[p] = Block{p, bytes, dev};
    }
    enum State { UNKNOWN, LIVE, IDLE };
    // LIVE: `b` is the caller's now, for put().
    State claim(void *p, size_t &bytes, int &dev) {
        std::lock_guard<std::mutex> lock(mu_);
        for (const Block &b : idle_)
            if (b.p == p) return IDLE;
        auto it = live_.find(p);
        if (it == live_.end()) return UNKNOWN;
        bytes = it->second.bytes;
        dev = it->second.dev;
        live_.erase(it);
        return LIVE;
    }
    // Keeps a block that no work uses any more; frees what that makes too much.  Throws (no host memory) before
    // anything has changed, or not at all: the caller then frees the block itself.
    hipError_t put(void *p, size_t bytes, int dev) {
        std::vector<Block> out;
        {
            std::lock_guard<std::mutex> lock(mu_);
            out.reserve(idle_.size() + 1);
            idle_.reserve(idle_.size() + 1);
            size_t avail = 0, total = 0;
            if (!limit_ && hipMemGetInfo(&avail, &total) == hipSuccess) limit_ = total / 64 + 1;
            if (bytes > limit_) {
                out.push_back(Block{p, bytes, dev});  // it alone: the smaller idle ones stay
            } else {
                idle_.push_back(Block{p, bytes, dev});
                held_ += bytes;
            }
            while (held_ > limit_ || idle_.size() > 64) {
                out.push_back(idle_.front());
                held_ -= idle_.front().bytes;
                idle_.erase(idle_.begin());
            }
        }
        return drop(out);
    }
    // Frees every idle block; false if there was none.
    bool release() {
        std::vector<Block> out;
        {
            std::lock_guard<std::mutex> lock(mu_);
            out.swap(idle_);
            held_ = 0;
        }
        (void)drop(out);
        return !out.empty();
    }

  private:
    struct Block {
        void *p;
        size_t bytes;
        int dev;
    };
    static hipError_t drop(const std::vector<Block> &out) {
        hipError_t e = hipSuccess;
        for (const Block &b : out) {
            const hipError_t f = hipFree(b.p);
            if (f != hipSuccess) e = f;
        }
        return e;
    }
    std::mutex mu_;
    std::map<void *, Block> live_;
    std::vector<Block> idle_;  // oldest first
    size_t held_ = 0, limit_ = 0;
};

}  // namespace omx
