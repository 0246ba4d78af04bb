// Launch selection of the split products (split_mm.hpp; the kernels are in
// k_split2/4/8.hip).
#include "split_mm.hpp"

namespace moehip {

static bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

bool split_supported(const WDesc &w, const float *x) {
    // whole units, and 16-byte loads of x, codes and scales
    return (w.bits == 2 || w.bits == 4 || w.bits == 8) && (w.type == 0 || w.type == 1 || w.type == 30) &&
           w.gshift >= 5 && w.gshift <= 7 && w.in % split::kUnit == 0 && aligned16(x) && aligned16(w.data) &&
           aligned16(w.scales) && aligned16(w.biases);
}

static hipError_t split_dispatch(const split::Launch &l, int mode) {
    switch (l.a.w.bits) {
    case 2: return split::launch2(l, mode);
    case 4: return split::launch4(l, mode);
    case 8: return split::launch8(l, mode);
    }
    return hipErrorInvalidValue;
}

// Where the split products overtake the VALU rows of k_batched.hip, which cost
// about one instruction per code and input row against a fixed cost per code:
//  - over dispatched segments, from 1.5 pairs an expert on average (0.75 at 8
//    bits, whose conversions the VALU rows repeat per input), amid the crossings
//    of three layers of h 2048.  A layer on VALU / split, us, at these pairs:
//      512 experts, ff 512: 2-bit 1.25 253 / 262, 1.5 291 / 278; 4-bit 1.25 232 /
//        242, 1.5 260 / 262, 1.75 285 / 273; 8-bit 0.47 185 / 187, 0.62 226 / 216
//      128 experts, ff 512: 2-bit 1.25 85.6 / 85.0, 1.5 95 / 97, 1.75 106 / 97;
//        4-bit 1.25 83 / 80, 1.5 88 / 90, 1.75 94 / 90; 8-bit (group 64) 0.5 71.5
//        / 73.2, 0.75 81.7 / 85.0, 1 94.8 / 93.4
//      128 experts, ff 768: 2-bit 1.5 117 / 120, 2 130 / 131, 2.5 149 / 138; 4-bit
//        1.25 101 / 105, 1.5 114 / 112; 8-bit 0.5 85.7 / 85.6, 0.75 108 / 107;
//  - over all tokens, from 96 rows: the shared expert's three products at 64 /
//    100 / 300 tokens 23 / 35 / 82 us against 25 / 26 / 38 on their own.
// Rows VALU does not take are split at any count (the grouped path instead: ff
// 640 at 1 / 2 / 8 tokens of 128 experts 73 / 115 / 209 us a layer, split 32 / 37
// / 64).
bool split_rows_better(const WDesc &w, uint32_t n, uint32_t experts) {
    if (experts <= 1) return n >= 96;
    return w.bits == 8 ? 4ull * n >= 3ull * experts : 2ull * n >= 3ull * experts;
}

hipError_t launch_split_gateup(Prof *p, hipStream_t s, const char *name, const WDesc &gate, const WDesc &up,
                               const float *x, const uint32_t *perm, uint32_t k, const uint32_t *tiles,
                               const uint32_t *ntiles, const uint32_t *offsets, uint32_t n, uint32_t entries,
                               float *act) {
    if (gate.bits != up.bits || gate.type != up.type || gate.gshift != up.gshift) return hipErrorInvalidValue;
    split::Args a{};
    a.w = gate;
    a.w2 = up;
    a.in = x;
    a.perm = perm;
    a.k = k;
    a.tiles = tiles;
    a.ntiles = ntiles;
    a.offsets = offsets;
    a.n = n;
    a.out = act;
    return split_dispatch(split::Launch{p, s, name, a, entries, 2}, split::GATEUP);
}

hipError_t launch_split_rows(Prof *p, hipStream_t s, const char *name, const WDesc &w, const float *in,
                             const uint32_t *tiles, const uint32_t *ntiles, const uint32_t *offsets, uint32_t n,
                             uint32_t entries, float *out) {
    // Two tiles a wave halve the input staging per weight row; one while that
    // leaves the grid within two blocks a CU, where only the length of a block's
    // own chain counts (h 2048 -> 4096 rows at 32 / 128 / 1000 rows of input:
    // 12 / 18 / 89 us with one tile, 17 / 18 / 76 with two).
    const uint64_t blocks1 = (uint64_t)((w.out + 63) / 64) * ((n + split::kRows - 1) / split::kRows);
    const int nt = !tiles && blocks1 <= 512 ? 1 : 2;
    // grid.y is limited to 65535 entries: longer runs of input rows in parts
    // (dispatched segments come with at most 65535 runs: block_entry sends more
    // to the grouped path)
    const uint32_t part = tiles ? n : 65535u * split::kRows;
    hipError_t e = hipSuccess;
    for (uint64_t n0 = 0; n0 < n && e == hipSuccess; n0 += part) {
        split::Args a{};
        a.w = w;
        a.w2 = w;
        a.in = in + n0 * w.in;
        a.tiles = tiles;
        a.ntiles = ntiles;
        a.offsets = offsets;
        a.n = (uint32_t)(n - n0 < part ? n - n0 : part);
        a.out = out + n0 * w.out;
        e = split_dispatch(split::Launch{p, s, name, a, entries, nt}, split::ROWS);
    }
    return e;
}

}  // namespace moehip
