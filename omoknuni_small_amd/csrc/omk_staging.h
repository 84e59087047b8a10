// Who may write where in the staging part of the pinned block (omk_api.hip): plain bookkeeping of the host, apart
// so that it can be tested without a GPU.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace omk {

// Staging is handed out front to back.  Kernels that have been enqueued read what was handed out, so it may start at
// the front again only once every one of them has run.  Two things show that: the stream is idle, or it has got as far
// as a point behind which nothing has been handed out.  Offsets do not show it: after a rewind the same offset comes
// back with other pieces on their way, which is why a point in time is the NUMBER of pieces handed out.
class Staging {
public:
    static constexpr size_t kFull = ~(size_t)0;

    explicit Staging(size_t room = 0) : room_(room) {}
    size_t room() const { return room_; }

    // `bytes`, rounded up to a cache line: their offset, or kFull when they do not fit behind what is in use
    size_t take(size_t bytes) {
        bytes = (bytes + 127) & ~(size_t)127;
        if (bytes > room_ - used_) return kFull;
        const size_t at = used_;
        used_ += bytes;
        handed_++;
        return at;
    }
    uint64_t now() const { return handed_; }
    // everything enqueued has run
    void idle() { used_ = 0; }
    // everything enqueued before `point` (a now()) has run
    void ran_to(uint64_t point) {
        if (point == handed_) used_ = 0;
    }

private:
    size_t room_, used_ = 0;
    uint64_t handed_ = 0;
};

}  // namespace omk
