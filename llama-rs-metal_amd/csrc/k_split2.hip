// The split products (split_mm.hpp) over 2-bit codes, in a translation unit
// of their own so the code widths compile beside each other.
#include "split_mm.hpp"

namespace moehip {

hipError_t split::launch2(const Launch &l, int mode) {
    return mode == GATEUP ? l.kind<GATEUP, 2>() : l.kind<ROWS, 2>();
}

}  // namespace moehip
