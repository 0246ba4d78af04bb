// F32-accurate products of F32 rows with affine weights on the f16 matrix
// cores (v_mfma_f32_16x16x32_f16), for segments of a few to a few dozen rows.
//
//   GATEUP  act[p, j] = silu(x_t . G_e[j]) * (x_t . U_e[j])   t = perm[p] / k
//           (activation, crates/metal-backend/src/shaders/elementwise.metal:8-17)
//   ROWS    out[p, r] = in_p . W_e[r]
//           (Batch::matmul, crates/metal-backend/src/apple/ops/matrix.rs:63-148;
//           expert_matmul(down), crates/model-runtime/src/execute.rs:225)
//
// Why it is exact enough: an affine weight is code * scale + bias with a code
// of at most 8 bits, and code - 2^(bits-1) is exact in f16.  An input value,
// scaled by a power of two per row and 128 values, is split into two f16
// terms hi + lo (hi rounded to nearest, lo the rounded remainder): off by at
// most 2^-22 of it (2^-24 on average), or, where that is smaller than lo's
// subnormal spacing, by 2^-39 of the largest of the 128.  So sum(code * x) over
// a quantization group is two matrix products whose single products are exact
// (their sum rounds in the F32 accumulator), and the group's scale and bias are
// applied to that sum in F32:
//   out = sum_g scale_g * D_g + (bias_g + 2^(bits-1) scale_g) * sum_g(x),
// a group's two terms first, so that the running sum rounds once per group.
// The centred codes and the one F32 addition per group leave it closer to the
// 64-bit product than a chain of F32 multiply-adds over the unsigned codes.
//
// What bounds it: a conversion per code (1.1 instructions) whatever the rows
// that share it, where the F32 dot of k_batched.hip costs one per code and row;
// then the memory pipe, whose loads gather 64 bytes from each of 16 rows.  512
// experts of h 2048, ff 512 (4-bit, group 64) at 500 tokens, 10 pairs an expert:
// gate/up 615 us on VALU, 196 here (3.1 TB/s of codes; without the products 157),
// down 411 -> 114.  h 2048 -> 4096 rows over 2000 tokens 144 us (233 TFLOP/s as
// F32), where the F32 matrix cores take 280.  Against 64 bits the products of
// 2048 values in groups of 64 are off by 1.4e-7, those of the F32 matrix cores
// by 8.1e-7.
// Entries of 32 and 64 rows, four tiles a wave, eight waves a block and codes
// four units ahead were all slower (fewer waves per SIMD; 26 to 60%).
//
// Block = 4 waves over one entry of at most 16 input rows and 64 * NT
// weight rows; wave w owns NT tiles of 16 weight rows (GATEUP: NT/2 of gate
// and the same outputs' NT/2 of up).  Per unit of 128 input values:
//   - the block's threads hold the next unit's x in registers (16 threads x 8
//     values a row), scale, split and store it to the idle LDS buffer with the
//     rows' scales and per-group sums; 16-byte chunks are XOR-swizzled by the
//     row, so the fragment reads (16 rows of one chunk) hit every bank once;
//   - each wave loads its codes straight into registers, one 16-byte (4-bit)
//     load per tile: lane (n, q) = (l % 16, l / 16) takes weight row n, values
//     32q .. 32q + 31, two units ahead.  A matrix instruction sums over 32
//     values, 8 from each q, which must lie in one quantization group:
//     v_permlane32_swap (group 64) and v_permlane16_swap (group 32) move the
//     words between the q rows until each fragment does; x is read from LDS in
//     the same order.
// One barrier per unit.
#pragma once
#include <type_traits>

#include "codes16.hpp"
#include "rowdot.hpp"

namespace moehip {

namespace split {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
using namespace codes16;

enum { GATEUP = 0, ROWS = 1 };

constexpr int kUnit = 128;             // input values per iteration
constexpr int kRows = 16;              // input rows per entry
constexpr int kWaves = 4, kThreads = 64 * kWaves;

struct Args {
    WDesc w, w2;              // weights (w2: the up rows of GATEUP)
    const float *in;          // input rows [*, w.in]
    const uint32_t *perm;     // GATEUP over dispatched pairs: input row perm[p] / k
    uint32_t k;
    const uint32_t *tiles;    // entries (expert, first p), or nullptr: runs over [0, n)
    const uint32_t *ntiles;   // entry count (device), with tiles
    const uint32_t *offsets;  // segment bounds [e], [e + 1], with tiles
    uint32_t n;               // without tiles: input rows
    float *out;               // [p, w.out]
};

// One buffer of the block's input rows for one unit.
struct Stage {
    uint8_t a[2][kRows][kUnit * 2];  // hi and lo terms, f16
    float sums[4][kRows];            // sums of the scaled x over 32 values, per group of 32
    float scale[kRows];              // 2^(e-15): a * scale = x
};

__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b) {
    const auto r = __builtin_amdgcn_permlane32_swap((int)a, (int)b, false, false);
    a = (uint32_t)r[0];
    b = (uint32_t)r[1];
}
__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b) {
    const auto r = __builtin_amdgcn_permlane16_swap((int)a, (int)b, false, false);
    a = (uint32_t)r[0];
    b = (uint32_t)r[1];
}

// The scales and biases of one lane's weight row for four units.  Lane row q
// loads those of unit 4v + q (one load of each per four units; a load per unit
// with every lane row reading the same words kept the memory pipe busier than
// the codes did: gate/up at 500 tokens 284 -> 157 us without it), and the swaps
// hand each unit's words to all lane rows.  T: the scales' type.
template <int T, int GS>
struct Scales {
    static constexpr int SZ = T == 0 ? 4 : 2;
    static constexpr int NG = kUnit >> GS;        // groups per unit
    static constexpr int NS = (NG * SZ + 3) / 4;  // words per unit
    uint32_t raw[2][NS];                 // [scales, biases], as loaded
    uint32_t even[2][NS], odd[2][NS];    // unit 0 | unit 2 in the lower | upper half, and 1 | 3

    __device__ __forceinline__ static void words(uint32_t *d, const void *base, uint64_t group) {
        const uint8_t *p = reinterpret_cast<const uint8_t *>(base) + group * SZ;
        if constexpr (NG * SZ == 2) {
            d[0] = *reinterpret_cast<const uint16_t *>(p);
        } else if constexpr (NS == 1) {
            d[0] = *reinterpret_cast<const uint32_t *>(p);
        } else if constexpr (NS == 2) {
            const u32x2 v = *reinterpret_cast<const u32x2 *>(p);
            d[0] = v[0];
            d[1] = v[1];
        } else {
            const u32x4 v = *reinterpret_cast<const u32x4 *>(p);
#pragma unroll
            for (int i = 0; i < 4; i++) d[i] = v[i];
        }
    }
    // el: element index of the weight row; unit: this lane row's unit
    __device__ __forceinline__ void load(const WDesc &wd, uint64_t el, uint32_t unit) {
        const uint64_t g = (el + unit * kUnit) >> GS;
        words(raw[0], wd.scales, g);
        words(raw[1], wd.biases, g);
    }
    __device__ __forceinline__ void spread() {
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
            for (int i = 0; i < NS; i++) {
                even[k][i] = odd[k][i] = raw[k][i];
                swap16(even[k][i], odd[k][i]);
            }
    }
    // unit j of the four: words k = 0 scales, 1 biases
    __device__ __forceinline__ void unit(int j, int k, uint32_t *d) const {
#pragma unroll
        for (int i = 0; i < NS; i++) {
            uint32_t lo = j & 1 ? odd[k][i] : even[k][i], hi = lo;
            swap32(lo, hi);
            d[i] = j < 2 ? lo : hi;
        }
    }
    // scale or bias of group g of the unit
    __device__ __forceinline__ static float value(const uint32_t *d, int g) {
        if constexpr (SZ == 4) return __uint_as_float(d[g]);
        else return raw_to_f32<T>((d[g >> 1] >> (16 * (g & 1))) & 0xffffu);
    }
};

// One lane's share of one 16-row tile and unit: 32 codes of its weight row.
template <int BITS, int GS>
struct Codes {
    uint32_t w[BITS];

    // el: element index of the weight row's first value of the unit
    __device__ __forceinline__ void load(const WDesc &wd, uint64_t el, int q) {
        const uint8_t *p = reinterpret_cast<const uint8_t *>(wd.data) + (el + 32 * q) * BITS / 8;
        if constexpr (BITS == 2) {
            const u32x2 v = *reinterpret_cast<const u32x2 *>(p);
            w[0] = v[0];
            w[1] = v[1];
        } else {
#pragma unroll
            for (int i = 0; i < BITS / 4; i++) {
                const u32x4 v = reinterpret_cast<const u32x4 *>(p)[i];
#pragma unroll
                for (int j = 0; j < 4; j++) w[4 * i + j] = v[j];
            }
        }
    }
    // Moves the words so that fragment i of every lane row q lies in one
    // group: fragments i of group 64: chunk 8 (i / 2) + 4 (q % 2) + 2 (q / 2)
    // + i % 2 of the unit, group 32: chunk 4i + q, group 128: chunk 4q + i
    // (chunk_of).
    __device__ __forceinline__ void arrange() {
        constexpr int F = BITS / 4;  // words per fragment (2-bit: two fragments a word)
        if constexpr (GS <= 6) {
            if constexpr (BITS == 2) {
                swap32(w[0], w[1]);
            } else {
#pragma unroll
                for (int i = 0; i < 2 * F; i++) swap32(w[i], w[i + 2 * F]);
            }
        }
        if constexpr (GS == 5) {
            if constexpr (BITS == 2) {
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    uint32_t lo = w[i], hi = w[i] >> 16;  // fragments 2i, 2i + 1
                    swap16(lo, hi);
                    w[i] = (lo & 0xffffu) | (hi << 16);
                }
            } else {
#pragma unroll
                for (int i = 0; i < F; i++) {
                    swap16(w[i], w[i + F]);
                    swap16(w[2 * F + i], w[3 * F + i]);
                }
            }
        }
    }
    __device__ __forceinline__ f16x8 frag(int i, const Magic &mg) const {
        if constexpr (BITS == 2) return code_frag<2>(w[i >> 1], 0, i & 1, mg);
        else if constexpr (BITS == 4) return code_frag<4>(w[i], 0, 0, mg);
        else return code_frag<8>(w[2 * i], w[2 * i + 1], 0, mg);
    }
};

template <int GS>
__device__ __forceinline__ int chunk_of(int i, int q) {
    if constexpr (GS == 6) return 8 * (i >> 1) + 4 * (q & 1) + 2 * (q >> 1) + (i & 1);
    else if constexpr (GS == 5) return 4 * i + q;
    else return 4 * q + i;
}

// Scales, splits and stores one thread's 8 values (chunk c of row r).
__device__ __forceinline__ void put_chunk(Stage &st, int r, int c, const float *v) {
    float m = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) m = fmaxf(m, fabsf(v[j]));
    // the row's largest magnitude over the unit (16 lanes)
    m = fmaxf(m, dpp_f<kDppQuad1>(m));
    m = fmaxf(m, dpp_f<kDppQuad2>(m));
    m = fmaxf(m, dpp_f<kDppHalfMirror>(m));
    m = fmaxf(m, dpp_f<kDppMirror>(m));
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) sum += v[j];
    // (a NaN, which fmaxf drops, and an infinity reach the row's products as
    // NaN, through hi and through lo = inf - inf; body() computes such outputs
    // again from decoded weights)
    sum += dpp_f<kDppQuad1>(sum);
    sum += dpp_f<kDppQuad2>(sum);
    // 2^e > m; clamped so that 2^(15-e) stays finite (rows below 2^-106 keep
    // an absolute error of 2^-130)
    const int e = max(__builtin_amdgcn_frexp_expf(m), -105);
    const float up = __builtin_amdgcn_ldexpf(1.0f, 15 - e);
    u32x4 hi, lo;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float x0 = v[j] * up, x1 = v[j + 4] * up;
        const f16x2 h = __builtin_convertvector((f32x2){x0, x1}, f16x2);
        hi[j] = as_u32(h);
        lo[j] = as_u32(__builtin_convertvector((f32x2){x0 - (float)h[0], x1 - (float)h[1]}, f16x2));
    }
    const int at = 16 * (c ^ (r & 15));
    *reinterpret_cast<u32x4 *>(&st.a[0][r][at]) = hi;
    *reinterpret_cast<u32x4 *>(&st.a[1][r][at]) = lo;
    if ((c & 3) == 0) st.sums[c >> 2][r] = sum * up;
    if (c == 0) st.scale[r] = __builtin_amdgcn_ldexpf(1.0f, e - 15);
}

// One output in F32 with its weights decoded first (code * scale + bias, two
// roundings, the values Tensor::decode produces), for results the split has no
// finite value for: an infinite input has no lo term (inf - inf), and inputs
// above about 2^122 can overflow the sum of a group's inputs.
// A lane's own loop over the row: such results are rare.
template <int BITS, int T>
__device__ __forceinline__ float decoded_dot(const WDesc &wd, uint64_t el, const float *x) {
    constexpr int P = 32 / BITS;
    const uint32_t *wp = reinterpret_cast<const uint32_t *>(wd.data) + el / P;
    float acc = 0.f;
#pragma unroll 1
    for (uint32_t k = 0; k < wd.in; k += P) {
        const uint64_t g = (el + k) >> wd.gshift;
        const float s = raw_to_f32<T>(load_raw<T>(wd.scales, g)), b = raw_to_f32<T>(load_raw<T>(wd.biases, g));
        float c[P];
        unpack_word<BITS>(wp[k / P], c);
#pragma unroll
        for (int j = 0; j < P; j++) {
            float w;
            {
#pragma clang fp contract(off)
                w = c[j] * s + b;
            }
            acc = fmaf(w, x[k + j], acc);
        }
    }
    return acc;
}

// Rows [beg, end) of the entry (at most kRows), weight rows of block column bx.
template <int MODE, int BITS, int T, int GS, int NT>
__device__ __forceinline__ void body(const Args &a, Stage *st, uint32_t bx, uint32_t e, uint32_t beg,
                                     uint32_t end) {
    static_assert(MODE == ROWS || NT % 2 == 0, "gate and up tiles pair up");
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n16 = lane & 15, q = lane >> 4;
    const uint32_t in = a.w.in, out = a.w.out, units = in / kUnit;
    Magic mg;
    mg.pin();
    // x: thread -> row tid / 16, chunk tid % 16 of the unit (rows past the end
    // repeat the first: a result row depends on its own input row only)
    const int xr = tid >> 4, xc = tid & 15;
    const uint32_t xpos = beg + xr < end ? beg + xr : beg;
    const uint32_t xsrc = MODE == GATEUP && a.perm ? a.perm[xpos] / a.k : xpos;
    const float *xp = a.in + (uint64_t)xsrc * in + 8 * xc;
    // weight rows: tile t, lane n16 (rows past `out` read row 0, never stored)
    constexpr int kOut = MODE == GATEUP ? NT / 2 : NT;  // output tiles per wave
    const uint32_t col0 = (bx * kWaves + wv) * (16 * kOut);
    uint64_t el[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        uint32_t r = col0 + 16 * (MODE == GATEUP ? t % kOut : t) + n16;
        if (r >= out) r = 0;
        el[t] = ((uint64_t)e * out + r) * in;
    }
    f32x4 xv[2];
    Codes<BITS, GS> cd[2][NT];
    Scales<T, GS> sc4[NT];
    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

    auto load_x = [&](uint32_t u) __attribute__((always_inline)) {
        const f32x4 *p = reinterpret_cast<const f32x4 *>(xp + u * kUnit);
        xv[0] = p[0];
        xv[1] = p[1];
    };
    auto put_x = [&](int buf) __attribute__((always_inline)) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = xv[j >> 2][j & 3];
        put_chunk(st[buf], xr, xc, v);
    };
    auto load_w = [&](int s, uint32_t u) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; t++) cd[s][t].load(MODE == GATEUP && t >= kOut ? a.w2 : a.w, el[t] + u * kUnit, q);
    };
    auto load_s = [&](uint32_t u) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; t++)
            sc4[t].load(MODE == GATEUP && t >= kOut ? a.w2 : a.w, el[t], min(u + (uint32_t)q, units - 1));
    };
    auto compute = [&](auto jc) __attribute__((always_inline)) {
        constexpr int J = decltype(jc)::value;  // unit of the four: register stage and LDS buffer J % 2
        constexpr int NG = kUnit >> GS, FG = 4 / NG;  // groups per unit, fragments per group
        const Stage &cur = st[J & 1];
#pragma unroll
        for (int t = 0; t < NT; t++) cd[J & 1][t].arrange();
        uint32_t sw[NT][2][Scales<T, GS>::NS];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            sc4[t].unit(J, 0, sw[t][0]);
            sc4[t].unit(J, 1, sw[t][1]);
        }
        const f32x4 fx = *reinterpret_cast<const f32x4 *>(&cur.scale[4 * q]);
#pragma unroll
        for (int g = 0; g < NG; g++) {
            f32x4 d[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) d[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int f = 0; f < FG; f++) {
                const int i = g * FG + f, at = 16 * (chunk_of<GS>(i, q) ^ n16);
                const f16x8 ah = *reinterpret_cast<const f16x8 *>(&cur.a[0][n16][at]);
                const f16x8 al = *reinterpret_cast<const f16x8 *>(&cur.a[1][n16][at]);
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const f16x8 c = cd[J & 1][t].frag(i, mg);
                    d[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, c, d[t], 0, 0, 0);
                    d[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, c, d[t], 0, 0, 0);
                }
            }
            // sums of the rows' scaled x over the group
            f32x4 xs = *reinterpret_cast<const f32x4 *>(&cur.sums[g * FG][4 * q]);
#pragma unroll
            for (int f = 1; f < FG; f++) {
                const f32x4 o = *reinterpret_cast<const f32x4 *>(&cur.sums[g * FG + f][4 * q]);
#pragma unroll
                for (int r = 0; r < 4; r++) xs[r] += o[r];
            }
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const float s = Scales<T, GS>::value(sw[t][0], g);
                const float b = fmaf((float)(1 << (BITS - 1)), s, Scales<T, GS>::value(sw[t][1], g));
#pragma unroll
                for (int r = 0; r < 4; r++) acc[t][r] = fmaf(fmaf(s, d[t][r], b * xs[r]), fx[r], acc[t][r]);
                // the group's sums are added here: left to itself the compiler
                // sinks every group's additions below the last one's products,
                // holding all their sums (half as many waves fit)
                asm volatile("" : "+v"(acc[t]));
            }
        }
    };
    // Unit u: multiply LDS buffer and code stage u % 2; store x of u + 1 (loaded
    // one unit earlier) into the other buffer, load x of u + 2 and the codes of
    // u + 2 into the registers just consumed; one barrier.  The scales of the
    // next four units load behind the first of these four.  Units past the last
    // are clamped (in bounds, unused).  Codes four units ahead cost more in
    // waves per SIMD than they hid (gate/up at 500 tokens 197 -> 203 us).
    const uint32_t last = units - 1;
    load_x(0);
    load_s(0);
    load_w(0, 0);
    load_w(1, min(1u, last));
    put_x(0);
    load_x(min(1u, last));
    __syncthreads();
    auto unit = [&](uint32_t u, auto jc) __attribute__((always_inline)) {
        constexpr int J = decltype(jc)::value;
        if constexpr (J == 0) {
#pragma unroll
            for (int t = 0; t < NT; t++) sc4[t].spread();
        }
        compute(jc);
        put_x((J + 1) & 1);
        load_x(min(u + 2, last));
        load_w(J & 1, min(u + 2, last));
        if constexpr (J == 0) load_s(min(u + 4, last));
        __syncthreads();
    };
    for (uint32_t u = 0; u < units; u += 4) {
        unit(u, std::integral_constant<int, 0>{});
        if (u + 1 < units) unit(u + 1, std::integral_constant<int, 1>{});
        if (u + 2 < units) unit(u + 2, std::integral_constant<int, 2>{});
        if (u + 3 < units) unit(u + 3, std::integral_constant<int, 3>{});
    }
    // acc[t][r]: input row 4 q + r, weight row 16 t + n16
    float bad = 0.f;  // NaN once an output is not finite
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const uint32_t p = beg + 4 * q + r;
        if (p >= end) continue;
#pragma unroll
        for (int t = 0; t < kOut; t++) {
            const uint32_t c = col0 + 16 * t + n16;
            if (c >= out) continue;
            float v = acc[t][r];
            if constexpr (MODE == GATEUP) v = v / (1.0f + expf(-v)) * acc[t + kOut][r];
            bad = fmaf(v, 0.f, bad);
            a.out[(uint64_t)p * out + c] = v;
        }
    }
    if (bad == 0.f) return;
#pragma unroll 1
    for (int i = 0; i < 4 * kOut; i++) {
        const uint32_t p = beg + 4 * q + i / kOut, c = col0 + 16 * (i % kOut) + n16;
        if (p >= end || c >= out) continue;
        float &o = a.out[(uint64_t)p * out + c];
        if (__builtin_isfinite(o)) continue;
        const uint64_t row = ((uint64_t)e * out + c) * in;
        const uint32_t src = MODE == GATEUP && a.perm ? a.perm[p] / a.k : p;
        const float *x = a.in + (uint64_t)src * in;
        float v = decoded_dot<BITS, T>(a.w, row, x);
        if constexpr (MODE == GATEUP) v = v / (1.0f + expf(-v)) * decoded_dot<BITS, T>(a.w2, row, x);
        o = v;
    }
}

// grid: x = weight-row blocks, y = entries.  Entries from the dispatch are its
// runs of 8 pairs: the block of every second run of a segment takes 16 pairs,
// the others exit.
template <int MODE, int BITS, int T, int GS, int NT>
__global__ __launch_bounds__(kThreads, 2) void split_kernel(Args a) {
    __shared__ __attribute__((aligned(16))) Stage st[2];
    uint32_t e = 0, beg, end;
    if (a.tiles) {
        if (blockIdx.y >= *a.ntiles) return;
        e = a.tiles[2 * blockIdx.y];
        beg = a.tiles[2 * blockIdx.y + 1];
        if ((beg - a.offsets[e]) % kRows) return;
        end = min(a.offsets[e + 1], beg + kRows);
    } else {
        beg = blockIdx.y * kRows;
        end = min(a.n, beg + kRows);
    }
    body<MODE, BITS, T, GS, NT>(a, st, blockIdx.x, e, beg, end);
}

struct Launch {
    Prof *p;
    hipStream_t s;
    const char *name;
    const Args &a;
    uint32_t entries;  // 8-pair runs (tiles), or 0: runs over a.n
    int nt;            // weight tiles per wave: 2, or (ROWS) 1
    template <int MODE, int BITS, int T, int GS, int NT>
    hipError_t go() const {
        const uint32_t cols = 16 * kWaves * (MODE == GATEUP ? NT / 2 : NT);
        const uint32_t ents = a.tiles ? entries : (a.n + kRows - 1) / kRows;
        return launch_kernel(p, name, split_kernel<MODE, BITS, T, GS, NT>,
                             dim3((a.w.out + cols - 1) / cols, ents), dim3(kThreads), 0, s, a);
    }
    template <int MODE, int BITS, int T, int GS>
    hipError_t tile() const {
        if constexpr (MODE == ROWS)
            if (nt == 1) return go<MODE, BITS, T, GS, 1>();
        return go<MODE, BITS, T, GS, 2>();
    }
    template <int MODE, int BITS>
    hipError_t kind() const {
        if (a.w.type == 0) return group<MODE, BITS, 0>();
        if (a.w.type == 1) return group<MODE, BITS, 1>();
        return group<MODE, BITS, 30>();
    }
    template <int MODE, int BITS, int T>
    hipError_t group() const {
        if (a.w.gshift == 5) return tile<MODE, BITS, T, 5>();
        if (a.w.gshift == 6) return tile<MODE, BITS, T, 6>();
        return tile<MODE, BITS, T, 7>();
    }
};

// k_split2/4/8.hip
hipError_t launch2(const Launch &l, int mode);
hipError_t launch4(const Launch &l, int mode);
hipError_t launch8(const Launch &l, int mode);

}  // namespace split

}  // namespace moehip
