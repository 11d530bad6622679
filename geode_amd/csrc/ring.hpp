// ring.hpp - slots used in turn (host code only, no other header).
#pragma once

namespace gv {

// The next of N slots, in turn, for as long as its owner lives: the slot itself is kept, always in [0, N), not a count of
// the uses (an int count passes 2^31 within a day of back-to-back calls, and the remainder of a negative one is negative).
template <int N>
struct Ring {
    int next = 0;
    int take() {
        const int s = next;
        next = s + 1 < N ? s + 1 : 0;
        return s;
    }
};

}  // namespace gv
