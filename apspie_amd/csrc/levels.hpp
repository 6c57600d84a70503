// A level loop whose host side follows the device without stopping it.  Each
// level's kernel reports that it began, in host memory, and the host keeps a
// few levels queued beyond that one; the kernel that finds nothing to do
// leaves the control block there too and says so.  A loop that launched
// chunks of 8, 16, 32, ... levels and waited for each drained the device at
// every chunk (20-25 us) and ran the rest of the last chunk empty (2 us a
// level): 116 of 249 launches for the 133 levels of a 2048^2 lattice.
#pragma once

#include "common.hpp"
#include "device.hpp"
#include "frontier.hpp"

namespace apspie {

class LevelFeed {
  public:
    // ahead: levels queued beyond the last one known to have begun
    LevelFeed(Ctx *c, int ahead)
        : c_(c), p_((Progress *)c->progress), ahead_((uint64_t)std::max(1, ahead)) {
        __atomic_store_n(&p_->started, (uint64_t)0, __ATOMIC_RELAXED);
        __atomic_store_n(&p_->done, (uint64_t)0, __ATOMIC_RELEASE);
    }
    // left by an exception: no kernel of this loop may report to the next one
    ~LevelFeed() {
        if (!finished_) (void)hipStreamSynchronize(c_->stream);
    }
    LevelFeed(const LevelFeed &) = delete;
    LevelFeed &operator=(const LevelFeed &) = delete;
    Progress *device() const { return p_; }
    // Waits until another level may be launched after `launched` ones; false
    // when the loop has ended.  The wait ends even if nothing is reported: a
    // stream found idle has no level left to wait for.
    bool more(int64_t launched) const {
        for (uint64_t spins = 0;; ++spins) {
            if (__atomic_load_n(&p_->done, __ATOMIC_ACQUIRE)) return false;
            if ((uint64_t)launched < __atomic_load_n(&p_->started, __ATOMIC_RELAXED) + ahead_)
                return true;
            if (spins % 16384 == 16383) {
                const hipError_t e = hipStreamQuery(c_->stream);
                if (e == hipSuccess) return !__atomic_load_n(&p_->done, __ATOMIC_ACQUIRE);
                if (e != hipErrorNotReady) APSPIE_HIP(e);
                (void)hipGetLastError();
            }
            __builtin_ia32_pause();
        }
    }
    // Waits for the stream (the call's end-of-call event: its timing ends
    // here) and returns the control block.
    const uint64_t *finish() {
        APSPIE_HIP(hipEventRecord(c_->ev1, c_->stream));
        APSPIE_HIP(hipEventSynchronize(c_->ev1));
        finished_ = true;
        c_->ev1_recorded = true;
        c_->stats.host_syncs++;
        return p_->ctl;
    }

  private:
    Ctx *c_;
    Progress *p_;
    uint64_t ahead_;
    bool finished_ = false;
};

// How far the host runs ahead: three levels by default, 3/8 of the option
// bfs_levels_per_sync.  Two to six measured the same within 1 % on long loops;
// each level more costs a short one the 2 us of another empty launch (R-MAT-14
// BFS: 72 / 74 / 75 / 78 / 84 us at 2 / 3 / 4 / 6 / 10).
inline int levels_ahead(Ctx *c) {
    return (int)std::max<int64_t>(1, opt(c, "bfs_levels_per_sync", 8) * 3 / 8);
}

}  // namespace apspie
