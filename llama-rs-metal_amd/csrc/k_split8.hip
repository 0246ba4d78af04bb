// The split products (split_mm.hpp) over 8-bit codes, in a translation unit
// of their own so the code widths compile beside each other.
#include "split_mm.hpp"

namespace moehip {

hipError_t split::launch8(const Launch &l, int mode) {
    return mode == GATEUP ? l.kind<GATEUP, 8>() : l.kind<ROWS, 8>();
}

}  // namespace moehip
