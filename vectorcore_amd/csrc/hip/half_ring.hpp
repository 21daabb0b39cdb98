// The bookkeeping of a ring of host memory that the GPU reads behind the host:
// two halves, each used from its start, and an event per half. Host code only.
#pragma once

#include <cstddef>

namespace vchip {

class HalfRing {
public:
    explicit HalfRing(std::size_t half_bytes) : half_bytes_(half_bytes) {}

    // The offset of the next n bytes (at most half_bytes). Bytes that do not fit the current half move the ring to
    // the other one: record(h) marks, in stream order, the end of what half h was used for, and wait(h) waits for
    // the last such mark, after which its bytes can be written again. State changes after a call that can fail.
    template <class Record, class Wait>
    std::size_t take(std::size_t n, Record&& record, Wait&& wait) {
        if (n > half_bytes_ - used_) {
            record(half_);
            recorded_[half_] = true;
            const int next = 1 - half_;
            if (recorded_[next]) wait(next);
            half_ = next;
            used_ = 0;
        }
        const std::size_t at = std::size_t(half_) * half_bytes_ + used_;
        used_ += n;
        return at;
    }

private:
    std::size_t half_bytes_;
    std::size_t used_ = 0;  // bytes of the current half
    int half_ = 0;
    bool recorded_[2] = {};
};

}  // namespace vchip
