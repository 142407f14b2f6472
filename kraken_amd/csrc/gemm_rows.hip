// gemm_rows.hip -- several activation rows against weights streamed once:
// dense GEMMs of 2..32 rows, and the routed experts' projections over their
// tokens.  The products are formed on the f16 matrix cores from the weight
// CODES, not from dequantized weights: a code of up to 8 bits is exact in
// f16, an f16 activation (or the two f16 planes of an f32 one) is exact too,
// so every product is exact, a 32-value sub-block's sum is rounded in f32
// only, and the block's scales enter in f32 (Q4_K: src/quant.cpp:427-447;
// Q5_K: 462-489; Q6_K: 491-512; Q8_0: 381-387; Q4_0: 331-339).
//
// Bound: HBM (every weight byte once); what is left beside it is one pass's
// ramp and tail (the preparation's launch, the first loads' latency, the
// waves' sums).  Measured, Q4_K f16 rows: 4096 -> 14336 8 rows 19.4 -> 16.0 us,
// 14336 -> 4096 8 rows 80.9 -> 20.8 us (6.7 us of HBM time each); the f16
// expert layer (128 experts, 4096 / 1536, top 8) 160 tokens 9797 -> 420 us.
// What the layout buys:
//   * A workgroup owns 16 or 32 weight rows over all of K; its waves split K
//     into contiguous slices of NBW 256-value blocks, and a wave requests
//     every weight byte of its slice before any arithmetic, so no barrier or
//     staging stands between the waves until their sums meet in LDS.
//   * One MFMA (16 activation rows x 16 weight rows x one sub-block) needs
//     the sub-block's 32 codes spread over the four 16-lane rows.  Weights
//     load 16 bytes a lane (the four lane rows cover whole 64-byte lines) and
//     cross-row lane swaps hand each row its share; the activations are
//     prepared in the order that leaves (rows_prep_kernel).
//   * Codes become f16 without conversions: a code placed in the mantissa of
//     1024 or 64 is 1024 + q or 64 + q, and one packed f16 operation takes the
//     constant off (with the sub-block's scale where scale x code is exact in
//     f16).  Left as subnormals they cost precision: the matrix cores take
//     them, but sums lose low bits (3.5e-6 against 2.7e-7).
//   * Q4_K / Q5_K minimums: one more MFMA per block, the 6-bit mins against
//     the activation rows' sub-block sums (three f16 planes, exact to 2^-33).
#include <cstdint>

#include "gemv_core.hpp"
#include "krk_mi355x.h"

namespace krk {

namespace {

typedef _Float16 h16x2 __attribute__((ext_vector_type(2)));

constexpr int kRowsWaves = 16;      // waves of a workgroup
constexpr int kRowsBlocks = 4;      // 256-value blocks of a wave's slice

constexpr bool has_min(int dt) { return dt == DT_Q4_K || dt == DT_Q5_K; }

// Where prepared rows lie.  A block of a row is nine 64-byte parts: its eight
// sub-blocks (four 16-byte pieces, one per lane row) and the sums.
//   Dense: sixteen rows interleaved piece by piece, so that one load of the
//   wave (16 rows x 4 pieces) is 1 KB in a row.  (Rows one after another put
//   the sixteen 64-byte parts of a load 9216 bytes apart, on a quarter of the
//   L2's channels: Q4_K 4096 -> 14336, 16 rows 18.8 -> 16.4 us, 32 rows 28.0
//   -> 22.2.)
//   Routed: the rows of an expert are any tokens', so each row on its own, an
//   odd number of 256-byte units apart, which spreads them over the channels.
template <bool DENSE> struct PrepAt {
    static constexpr int kPart = DENSE ? 1024 : 64, kPiece = DENSE ? 256 : 16, kBlock = 9 * kPart;
    __host__ __device__ static int64_t stride(int nb) {   // bytes of sixteen rows / of a row
        return DENSE ? static_cast<int64_t>(nb) * kBlock : ((static_cast<int64_t>(nb) * kBlock + 255) / 256 | 1) * 256;
    }
    __device__ static int64_t row(int64_t r, int nb) {
        return DENSE ? (r >> 4) * stride(nb) + (r & 15) * 16 : r * stride(nb);
    }
};

// the first code byte (of a 32-code run) that lane row g holds after the
// half-wave swap of two 16-byte pieces: 0, 16, 8, 24
__device__ __forceinline__ int lane_base(int g) { return 16 * (g & 1) + 8 * (g >> 1); }
// the dword (of a 16-byte run) that lane row g holds after the 4 x 4
// transpose below: 0, 2, 1, 3
__device__ __forceinline__ int lane_dword(int g) { return 2 * (g & 1) + (g >> 1); }

__device__ __forceinline__ void swap32(uint32_t a, uint32_t b, uint32_t &lo, uint32_t &hi) {
    const auto s = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    lo = s[0];
    hi = s[1];
}
__device__ __forceinline__ void swap16(uint32_t a, uint32_t b, uint32_t &lo, uint32_t &hi) {
    const auto s = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    lo = s[0];
    hi = s[1];
}
// lane rows hold four dwords each; afterwards p[t] holds, in lane row g,
// dword lane_dword(g) of lane row t
__device__ __forceinline__ void transpose4(const u32x4 &v, uint32_t (&p)[4]) {
    uint32_t a, b, c, e;
    swap32(v.x, v.y, a, b);
    swap32(v.z, v.w, c, e);
    swap16(a, c, p[0], p[1]);
    swap16(b, e, p[2], p[3]);
}
// lane row R's value, in every lane row
template <int R> __device__ __forceinline__ uint32_t lane_row(uint32_t v) {
    uint32_t a, b, c, e;
    swap32(v, v, a, b);
    const uint32_t w = R < 2 ? a : b;
    swap16(w, w, c, e);
    return (R & 1) ? e : c;
}

// bytes 2h, 2h + 1 of w as the f16 pair (1024 + b): 0x64 is 1024's high byte
template <int H> __device__ __forceinline__ h16x2 bytes_f16(uint32_t w) {
    return __builtin_bit_cast(h16x2, __builtin_amdgcn_perm(0x64646464u, w, H ? 0x04030402u : 0x04010400u));
}
__device__ __forceinline__ uint32_t add2(h16x2 v, float c) {
    const _Float16 h = static_cast<_Float16>(c);
    return __builtin_bit_cast(uint32_t, v + h16x2{h, h});
}
// The exponents codes go under and the masks that cut them out, kept in
// vector and scalar registers: as literals every (w & mask) | under would take
// two operations, for one that takes no literal and one scalar operand.  (The
// empty statements only hide the values from the compiler.)
struct Masks {
    uint32_t k1024 = 0x64006400u, k64 = 0x54005400u;               // 1024 and 64 in both halves
    uint32_t lo4 = 0x000F000Fu, hi4 = 0x00F000F0u, b8 = 0x00FF00FFu, n4 = 0x0F0F0F0Fu;
    __device__ __forceinline__ Masks() {
        asm("" : "+v"(k1024), "+v"(k64));
        asm("" : "+s"(lo4), "+s"(hi4), "+s"(b8), "+s"(n4));
    }
};
// A code under an f16 exponent is its value plus a bias (1024 + q: ulp 1, bits
// 0..9; 64 + q: ulp 1/16, bits 4..7), which a packed f16 operation takes off
// exactly.  (As f16 subnormals codes would need no bias, and the matrix cores
// take those, but the low bits of the products' sums are then lost: 3.5e-6
// against 2.7e-7 relative, f32 rows.)
//
// v c + o on both halves
__device__ __forceinline__ uint32_t fma2(uint32_t v, _Float16 c, _Float16 o) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(h16x2, v), h16x2{c, c}, h16x2{o, o}));
}
template <int K> __device__ __forceinline__ float sbyte(uint32_t w) {
    return static_cast<float>(static_cast<int32_t>(w << (24 - 8 * K)) >> 24);
}

__device__ __forceinline__ half8 as_half8(const u32x4 &v) { return __builtin_bit_cast(half8, v); }
__device__ __forceinline__ half8 as_half8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(half8, u32x4{a, b, c, d});
}
__device__ __forceinline__ floatx4 mfma32(const u32x4 &a, const half8 &b, const floatx4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(as_half8(a), b, c, 0, 0, 0);
}
#define KRK_ZERO4 (floatx4{0.0f, 0.0f, 0.0f, 0.0f})

// acc += c v, component by component
__device__ __forceinline__ void axpy(floatx4 &acc, float c, const floatx4 &v) {
#pragma unroll
    for (int r = 0; r < 4; r++) acc[r] = __builtin_fmaf(c, v[r], acc[r]);
}

// the 6-bit scales and mins of Q4_K / Q5_K (get_scale_min_k4,
// src/quant.cpp:427-435) as bytes, from the block's 16-byte header
template <int S> __device__ __forceinline__ _Float16 k_scale(const u32x4 &h) {
    const uint32_t b = S < 4 ? h.y & 0x3F3F3F3Fu : (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u);
    return static_cast<_Float16>(static_cast<uint16_t>((b >> (8 * (S & 3))) & 63u));
}
// the mins in f16, sub-blocks 0 2 1 3 4 6 5 7
__device__ __forceinline__ half8 k_mins(const u32x4 &h, const Masks &k) {
    const uint32_t m0 = h.z & 0x3F3F3F3Fu, m1 = ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u);
    auto f = [&](uint32_t w) { return add2(__builtin_bit_cast(h16x2, (w & k.b8) | k.k1024), -1024.0f); };
    return as_half8(f(m0), f(m0 >> 8), f(m1), f(m1 >> 8));
}

// keeps what is computed from v inside the loop it stands in: the codes built
// from a block serve one pass over the rows, and built ahead for all passes
// they would need several times the registers of the block's own bytes
__device__ __forceinline__ void pin(uint32_t &v) { asm volatile("" : "+v"(v)); }
template <typename V> __device__ __forceinline__ void pin(V &v) {
    constexpr int N = sizeof(V) / 4;
#pragma unroll
    for (int i = 0; i < N; i++) {
        uint32_t w = v[i];
        pin(w);
        v[i] = w;
    }
}

// an accumulator's value is due here: without it the folds of several pairs
// are put off, and their MFMA results held in registers meanwhile
__device__ __forceinline__ void settle_acc(floatx4 &v) { asm volatile("" : "+v"(v)); }

// ---- one lane's share of one 256-value block of one weight row.  fetch()
// loads it; settle() hands the codes to the lane rows their sub-blocks need,
// in place; pair<P>() multiplies sub-blocks 2 P and 2 P + 1 with 16 prepared
// activation rows (x: the pair's fragments) into the block's sum t, or where
// its scales do not multiply the codes exactly into acc, and finish() takes
// the block's sum and minimums (xs: the rows' sub-block sums) to acc.
template <int DT> struct RowBlk;

template <> struct RowBlk<DT_Q4_K> {
    static constexpr int BB = 144;
    u32x4 h, q[2];
    __device__ __forceinline__ void hold() { pin(h); pin(q[0]); pin(q[1]); }
    __device__ __forceinline__ void fetch(gbyte *p, int g) {
        h = ld128(p);
        q[0] = ld128(p + 16 + 16 * g);
        q[1] = ld128(p + 80 + 16 * g);
    }
    __device__ __forceinline__ void settle() {   // pair 2 i at x, y of q[i], pair 2 i + 1 at z, w
#pragma unroll
        for (int i = 0; i < 2; i++) {
            uint32_t l0, h0, l1, h1;
            swap32(q[i].x, q[i].z, l0, h0);
            swap32(q[i].y, q[i].w, l1, h1);
            q[i] = u32x4{l0, l1, h0, h1};
        }
    }
    // scale x code, at most 63 x 15, is exact in f16, so the sub-blocks of a
    // block add up in the matrix cores
    template <int P> __device__ __forceinline__ void pair(const u32x4 (&x)[2], const Masks &k, floatx4 &t, floatx4 &) const {
        const u32x4 &v = q[P >> 1];
        const uint32_t w0 = (P & 1) ? v.z : v.x, w1 = (P & 1) ? v.w : v.y;
        const uint32_t s0 = w0 >> 8, s1 = w1 >> 8;
        const _Float16 se = k_scale<2 * P>(h), so = k_scale<2 * P + 1>(h);
        const _Float16 be = se * static_cast<_Float16>(-1024.0f), bo = so * static_cast<_Float16>(-64.0f);
        auto lo = [&](uint32_t w) { return fma2((w & k.lo4) | k.k1024, se, be); };
        auto hi = [&](uint32_t w) { return fma2((w & k.hi4) | k.k64, so, bo); };
        t = mfma32(x[0], as_half8(lo(w0), lo(s0), lo(w1), lo(s1)), t);
        t = mfma32(x[1], as_half8(hi(w0), hi(s0), hi(w1), hi(s1)), t);
    }
    __device__ __forceinline__ void finish(const u32x4 &xs, const Masks &k, const floatx4 &t, floatx4 &acc) const {
        axpy(acc, h2f(h.x & 0xFFFFu), t);
        axpy(acc, -h2f(h.x >> 16), mfma32(xs, k_mins(h, k), KRK_ZERO4));
    }
};

template <> struct RowBlk<DT_Q5_K> {
    static constexpr int BB = 176;
    u32x4 h, q[2];
    u32x2 b;   // the high-bit bytes of this lane's code positions
    __device__ __forceinline__ void hold() { pin(h); pin(q[0]); pin(q[1]); pin(b); }
    __device__ __forceinline__ void fetch(gbyte *p, int g) {
        h = ld128(p);
        b = *(const __attribute__((address_space(1))) u32x2 *)(p + 16 + lane_base(g));
        q[0] = ld128(p + 48 + 16 * g);
        q[1] = ld128(p + 112 + 16 * g);
    }
    __device__ __forceinline__ void settle() {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            uint32_t l0, h0, l1, h1;
            swap32(q[i].x, q[i].z, l0, h0);
            swap32(q[i].y, q[i].w, l1, h1);
            q[i] = u32x4{l0, l1, h0, h1};
        }
    }
    // codes of sub-block C: nibbles | bit C of the high-bit bytes at bit 4;
    // scale x code, at most 63 x 31, is exact in f16
    template <int C> __device__ __forceinline__ half8 codes(const Masks &k) const {
        constexpr int P = C >> 1;
        const u32x4 &v = q[P >> 1];
        uint32_t w0 = (P & 1) ? v.z : v.x, w1 = (P & 1) ? v.w : v.y;
        if (C & 1) { w0 >>= 4; w1 >>= 4; }
        const uint32_t b0 = (C < 4 ? b.x << (4 - C) : b.x >> (C - 4)) & 0x10101010u;
        const uint32_t b1 = (C < 4 ? b.y << (4 - C) : b.y >> (C - 4)) & 0x10101010u;
        const uint32_t c0 = (w0 & k.n4) | b0, c1 = (w1 & k.n4) | b1;
        const _Float16 sc = k_scale<C>(h);
        const _Float16 o = sc * static_cast<_Float16>(-1024.0f);
        auto f = [&](uint32_t w) { return fma2((w & k.b8) | k.k1024, sc, o); };
        return as_half8(f(c0), f(c0 >> 8), f(c1), f(c1 >> 8));
    }
    template <int P> __device__ __forceinline__ void pair(const u32x4 (&x)[2], const Masks &k, floatx4 &t, floatx4 &) const {
        t = mfma32(x[0], codes<2 * P>(k), t);
        t = mfma32(x[1], codes<2 * P + 1>(k), t);
    }
    __device__ __forceinline__ void finish(const u32x4 &xs, const Masks &k, const floatx4 &t, floatx4 &acc) const {
        axpy(acc, h2f(h.x & 0xFFFFu), t);
        axpy(acc, -h2f(h.x >> 16), mfma32(xs, k_mins(h, k), KRK_ZERO4));
    }
};

// Q6_K: scales per 16 values, so one 16 x 16 x 16 MFMA per group; lane row g
// holds four codes of every group, q - 32 exact in f16
template <> struct RowBlk<DT_Q6_K> {
    static constexpr int BB = 210;
    u32x4 l[2], s;
    u32x2 q[2];
    uint32_t dw;
    __device__ __forceinline__ void hold() { pin(l[0]); pin(l[1]); pin(q[0]); pin(q[1]); pin(s); pin(dw); }
    __device__ __forceinline__ void fetch(gbyte *p, int g) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            l[h] = ld128_a2(p + 64 * h + 16 * g);
            q[h] = u32x2{ld32_a2(p + 128 + 32 * h + 8 * g), ld32_a2(p + 132 + 32 * h + 8 * g)};
        }
        s = ld128_a2(p + 192);
        dw = ld16g(p + 208);
    }
    __device__ __forceinline__ void settle() {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t p[4], a, c;
            transpose4(l[h], p);
            l[h] = u32x4{p[0], p[1], p[2], p[3]};
            swap32(q[h].x, q[h].y, a, c);
            q[h] = u32x2{a, c};
        }
    }
    template <int C, int E> __device__ __forceinline__ void group(const u32x4 (&x)[2], const Masks &k, floatx4 &acc) const {
        constexpr int H = C >> 2, QD = C & 3, GI = 8 * H + 2 * QD + E, T = 2 * (QD & 1) + E;
        const u32x4 &v = l[H];
        const uint32_t w = T == 0 ? v.x : T == 1 ? v.y : T == 2 ? v.z : v.w, u = E ? q[H].y : q[H].x;
        const uint32_t c = ((QD < 2 ? w : w >> 4) & k.n4) |
                           ((QD < 2 ? u << (4 - 2 * QD) : u >> (2 * QD - 4)) & 0x30303030u);
        const half4 b = __builtin_bit_cast(half4, u32x2{add2(bytes_f16<0>(c), -1056.0f), add2(bytes_f16<1>(c), -1056.0f)});
        const uint32_t sv = GI < 4 ? s.x : GI < 8 ? s.y : GI < 12 ? s.z : s.w;
        const float ds = h2f(dw) * sbyte<GI & 3>(sv);
        const u32x4 &xv = x[C & 1];
        const half4 av = __builtin_bit_cast(half4, E ? u32x2{xv.z, xv.w} : u32x2{xv.x, xv.y});
        axpy(acc, ds, __builtin_amdgcn_mfma_f32_16x16x16f16(av, b, KRK_ZERO4, 0, 0, 0));
    }
    template <int P> __device__ __forceinline__ void pair(const u32x4 (&x)[2], const Masks &k, floatx4 &, floatx4 &acc) const {
        group<2 * P, 0>(x, k, acc);
        group<2 * P, 1>(x, k, acc);
        group<2 * P + 1, 0>(x, k, acc);
        group<2 * P + 1, 1>(x, k, acc);
    }
    __device__ __forceinline__ void finish(const u32x4 &, const Masks &, const floatx4 &, floatx4 &) const {}
};

template <> struct RowBlk<DT_Q8_0> {
    static constexpr int BB = 272;
    u32x4 v[4];
    uint32_t dw;   // d of blocks 2g (low half) and 2g + 1 of the eight
    __device__ __forceinline__ void hold() { pin(v[0]); pin(v[1]); pin(v[2]); pin(v[3]); pin(dw); }
    __device__ __forceinline__ void fetch(gbyte *p, int g) {
#pragma unroll
        for (int t = 0; t < 4; t++) v[t] = ld128_a2(p + 68 * t + 34 * (g >> 1) + 2 + 16 * (g & 1));
        dw = ld16g(p + 68 * g) | (ld16g(p + 68 * g + 34) << 16);
    }
    __device__ __forceinline__ void settle() {   // block 2 t at x, y of v[t], block 2 t + 1 at z, w
#pragma unroll
        for (int t = 0; t < 4; t++) {
            uint32_t l0, h0, l1, h1;
            swap32(v[t].x, v[t].z, l0, h0);
            swap32(v[t].y, v[t].w, l1, h1);
            v[t] = u32x4{l0, l1, h0, h1};
        }
    }
    __device__ __forceinline__ static half8 codes(uint32_t w0, uint32_t w1) {
        const uint32_t u0 = w0 ^ 0x80808080u, u1 = w1 ^ 0x80808080u;
        return as_half8(add2(bytes_f16<0>(u0), -1152.0f), add2(bytes_f16<1>(u0), -1152.0f),
                        add2(bytes_f16<0>(u1), -1152.0f), add2(bytes_f16<1>(u1), -1152.0f));
    }
    template <int P> __device__ __forceinline__ void pair(const u32x4 (&x)[2], const Masks &k, floatx4 &, floatx4 &acc) const {
        const uint32_t dp = lane_row<P>(dw);
        const half8 e = codes(v[P].x, v[P].y), o = codes(v[P].z, v[P].w);
        const floatx4 ce = mfma32(x[0], e, KRK_ZERO4), co = mfma32(x[1], o, KRK_ZERO4);
        axpy(acc, h2f(dp & 0xFFFFu), ce);
        axpy(acc, h2f(dp >> 16), co);
    }
    __device__ __forceinline__ void finish(const u32x4 &, const Masks &, const floatx4 &, floatx4 &) const {}
};

template <> struct RowBlk<DT_Q4_0> {
    static constexpr int BB = 144;
    u32x4 v[2];
    uint32_t dw;   // d of blocks g (low half) and 4 + g of the eight
    __device__ __forceinline__ void hold() { pin(v[0]); pin(v[1]); pin(dw); }
    __device__ __forceinline__ void fetch(gbyte *p, int g) {
#pragma unroll
        for (int t = 0; t < 2; t++) v[t] = ld128_a2(p + 18 * (4 * t + g) + 2);
        dw = ld16g(p + 18 * g) | (ld16g(p + 18 * (4 + g)) << 16);
    }
    __device__ __forceinline__ void settle() {   // block 4 t + s at component s of v[t]
#pragma unroll
        for (int t = 0; t < 2; t++) {
            uint32_t p[4];
            transpose4(v[t], p);
            v[t] = u32x4{p[0], p[1], p[2], p[3]};
        }
    }
    // nibbles as 1024 + q (bits 0..3) and 64 + q (bits 4..7), less the bias
    // and the format's 8
    __device__ __forceinline__ static half8 codes(uint32_t w, const Masks &k) {
        const uint32_t s = w >> 8;
        auto lo = [&](uint32_t u) { return add2(__builtin_bit_cast(h16x2, (u & k.lo4) | k.k1024), -1032.0f); };
        auto hi = [&](uint32_t u) { return add2(__builtin_bit_cast(h16x2, (u & k.hi4) | k.k64), -72.0f); };
        return as_half8(lo(w), lo(s), hi(w), hi(s));
    }
    template <int P> __device__ __forceinline__ void pair(const u32x4 (&x)[2], const Masks &k, floatx4 &, floatx4 &acc) const {
        const u32x4 &u = v[P >> 1];
        const half8 e = codes((P & 1) ? u.z : u.x, k), o = codes((P & 1) ? u.w : u.y, k);
        const uint32_t d0 = lane_row<2 * (P & 1)>(dw), d1 = lane_row<2 * (P & 1) + 1>(dw);
        const float de = h2f(P < 2 ? d0 & 0xFFFFu : d0 >> 16), dod = h2f(P < 2 ? d1 & 0xFFFFu : d1 >> 16);
        const floatx4 ce = mfma32(x[0], e, KRK_ZERO4), co = mfma32(x[1], o, KRK_ZERO4);
        axpy(acc, de, ce);
        axpy(acc, dod, co);
    }
    __device__ __forceinline__ void finish(const u32x4 &, const Masks &, const floatx4 &, floatx4 &) const {}
};

// value index within a 32-value sub-block (Q6_K: within its two groups) of
// prepared position (g, e): the order RowBlk's codes come in
template <int DT> __device__ __forceinline__ int prep_value(int g, int e) {
    if constexpr (DT == DT_Q4_K || DT == DT_Q5_K)
        return lane_base(g) + (e & 4) + (((e & 1) << 1) | ((e >> 1) & 1));
    else if constexpr (DT == DT_Q8_0)
        return lane_base(g) + e;
    else if constexpr (DT == DT_Q6_K)
        return 16 * (e >> 2) + 4 * lane_dword(g) + (e & 3);
    else
        return 16 * (e >> 2) + 4 * lane_dword(g) + (((e & 1) << 1) | ((e >> 1) & 1));
}

__device__ __forceinline__ float dpp_xor1(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
}
__device__ __forceinline__ float dpp_xor2(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false));
}

// An activation row prepared for RowBlk: scaled by the power of two that
// brings its largest magnitude into [2^9, 2^10) (so a sub-block's sum stays
// within f16), as one f16 plane (f16 activations: exact; f32 ones rounded,
// where the caller's path allows f16 operands) or two (hi + lo, exact to
// 2^-23 of the value or 2^-35 of the row's largest), the 16-byte pieces of a
// sub-block in RowBlk's order, and for formats with mins the sub-block sums
// as three f16 planes.  inv[row] undoes the scale.  A row that holds a
// non-finite value is not scaled, and comes out non-finite.
// Grid: (rows, slices of 32 blocks); every workgroup finds the row's maximum
// for itself.
// Two planes, dense: rows 0..7 of sixteen are the hi planes of eight rows,
// 8..15 their lo planes; routed: row 2 r is the hi plane of row r, 2 r + 1 its
// lo plane.
template <int DT, typename XT, bool DENSE>
__global__ void __launch_bounds__(256) rows_prep_kernel(const XT *__restrict__ x, int64_t x_stride, int nb,
                                                        int planes, const int32_t *__restrict__ n_rows,
                                                        uint8_t *__restrict__ xp, float *__restrict__ inv) {
    __shared__ float wmax[4];
    const int64_t row = blockIdx.x;
    if (n_rows && row >= *n_rows) return;
    const XT *xr = x + row * x_stride;
    const int tid = threadIdx.x;
    float mx = 0.0f;
    bool nan = false;
    for (int i = 8 * tid; i < 256 * nb; i += 2048) {
        float v[8];
        load_run<8>(xr + i, v);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            mx = fmaxf(mx, fabsf(v[k]));
            nan |= v[k] != v[k];
        }
    }
    if (nan) mx = __builtin_inff();
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) mx = fmaxf(mx, shfl_xor(mx, m));
    if ((tid & 63) == 0) wmax[tid >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    const int eb = static_cast<int>((__float_as_uint(mx) >> 23) & 255u);
    int k = mx > 0.0f && eb < 255 ? 136 - eb : 0;
    k = k > 126 ? 126 : k;
    const float up = __uint_as_float(static_cast<uint32_t>(127 + k) << 23);
    if (tid == 0 && blockIdx.y == 0) inv[row] = __uint_as_float(static_cast<uint32_t>(127 - k) << 23);
    using At = PrepAt<DENSE>;
    uint8_t *out = xp + At::row(planes == 2 ? (DENSE ? 16 * (row >> 3) + (row & 7) : 2 * row) : row, nb);
    const int64_t lo_at = DENSE ? 8 * 16 : At::stride(nb);   // the lo plane's row, from the hi plane's
    const int units = 32 * nb, u0 = static_cast<int>(blockIdx.y) * 1024;
    for (int u = u0 + tid; u < units && u < u0 + 1024; u += 256) {
        const int blk = u >> 5, s = (u >> 2) & 7, g = u & 3;
        const XT *src = xr + 256 * blk + 32 * s;
        half8 hi, lo;
        float sum = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float v = static_cast<float>(src[prep_value<DT>(g, e)]) * up;
            hi[e] = static_cast<_Float16>(v);
            const float r = v - static_cast<float>(hi[e]);
            lo[e] = static_cast<_Float16>(r);
            sum += planes == 2 ? v : static_cast<float>(hi[e]);
        }
        uint8_t *o = out + static_cast<int64_t>(blk) * At::kBlock + At::kPiece * g;
        *reinterpret_cast<half8 *>(o + At::kPart * s) = hi;
        if (planes == 2) *reinterpret_cast<half8 *>(o + lo_at + At::kPart * s) = lo;
        if constexpr (has_min(DT)) {
            // lane g of the quad writes plane g of the sub-block's sum, at the
            // place its min takes (0 2 1 3 4 6 5 7)
            sum += dpp_xor1(sum);
            sum += dpp_xor2(sum);
            const _Float16 p0 = static_cast<_Float16>(sum);
            const float r1 = sum - static_cast<float>(p0);
            const _Float16 p1 = static_cast<_Float16>(r1);
            const _Float16 p2 = static_cast<_Float16>(r1 - static_cast<float>(p1));
            const _Float16 z = static_cast<_Float16>(0.0f);
            const int at = At::kPart * 8 + 2 * ((s & 4) | ((s & 1) << 1) | ((s >> 1) & 1));
            *reinterpret_cast<_Float16 *>(o + at) = g == 0 ? p0 : g == 1 ? p1 : g == 2 ? p2 : z;
            if (planes == 2) *reinterpret_cast<_Float16 *>(o + lo_at + at) = z;
        }
    }
}

// One output's sums of the waves, in wave order (at: wave 0's, `wave` floats
// apart; two planes: the lo plane's row lies `lo` floats on).  NWX: exactly
// NWMAX waves, which lets the reads all be in flight.
template <int NWMAX, bool NWX>
__device__ __forceinline__ float wave_sums(const float *at, int wave, int lo, int nw, int planes) {
    float v = 0.0f;
    if (planes == 2) {
#pragma unroll
        for (int q = 0; q < NWMAX; q++)
            if (NWX || q < nw) v += at[q * wave] + at[q * wave + lo];
    } else {
#pragma unroll
        for (int q = 0; q < NWMAX; q++)
            if (NWX || q < nw) v += at[q * wave];
    }
    return v;
}

// Dense.  One workgroup: weight rows [n0, n0 + 16 RG) of a segment over the
// blocks of K range blockIdx.z, one a wave, against all activation rows, 16
// prepared rows a pass.
template <int DT, int RG, int NWMAX, bool NWX>
__global__ void __launch_bounds__(64 * NWMAX) __attribute__((amdgpu_waves_per_eu(4))) rows_kernel(RowsArgs a) {
    extern __shared__ __align__(16) float red[];
    constexpr int S = 16 * RG + 4;          // red row stride: the four lane rows' stores spread over the banks
    using At = PrepAt<true>;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = NWX ? NWMAX : static_cast<int>(blockDim.x) >> 6;
    const int j = lane & 15, g = lane >> 4;
    const int kz = static_cast<int>(blockIdx.z) * a.range;   // this K range's first block
    const int kend = kz + a.range < a.nb ? kz + a.range : a.nb;
    const int blk = kz + wv;
    const bool live = blk < kend;           // (a range shorter than the others leaves its last wave idle)
    const RowsSeg &sg = a.seg[blockIdx.y];
    void *out = sg.out;
    const int64_t n_out = sg.n_out;
    constexpr int rows_sh = RG == 4 ? 6 : RG == 2 ? 5 : 4, rows_t = 1 << rows_sh;
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * rows_t;
    if (n0 >= n_out) return;                // a segment shorter than the grid's width
    const int per = a.planes == 2 ? 8 : 16;             // rows a pass

    // the pass's prepared rows (sixteen; those past the last hold whatever was
    // there, and their results go nowhere).  Once a pair of sub-blocks is
    // multiplied, its registers take the same pair of the next pass.
    gbyte *xrow = to_global(a.xp) + At::row(j, a.nb) + static_cast<int64_t>(blk) * At::kBlock + At::kPiece * g;
    u32x4 xa[4][2], xs = {0u, 0u, 0u, 0u};
    auto load_pair = [&](int p) {
#pragma unroll
        for (int s = 0; s < 2; s++) xa[p][s] = ld128(xrow + At::kPart * (2 * p + s));
    };
    auto load_sums = [&]() {
        if constexpr (has_min(DT)) xs = ld128(xrow + At::kPart * 8);
    };
    const Masks masks;
    RowBlk<DT> wr[RG];
    if (live) {
#pragma unroll
        for (int p = 0; p < 4; p++) load_pair(p);
        load_sums();
        // every weight byte of the wave's block of the tile
#pragma unroll
        for (int r = 0; r < RG; r++) {
            int64_t n = n0 + 16 * r + j;
            n = n < n_out ? n : n_out - 1;
            wr[r].fetch(to_global(sg.w + n * a.row_bytes) + static_cast<int64_t>(blk) * RowBlk<DT>::BB, g);
        }
    }

    const int64_t prow = static_cast<int64_t>(a.rows) * a.part_n;   // floats of one K range's partials
    for (int p0 = 0; p0 < a.rows; p0 += per) {
        const bool more = p0 + per < a.rows;
        floatx4 acc[RG];
#pragma unroll
        for (int r = 0; r < RG; r++) acc[r] = KRK_ZERO4;
        if (live) {
            if (more) xrow += At::stride(a.nb);
            // row group by row group, in the order they were requested: a
            // group is multiplied while the next ones are still on their way
            // (the scheduling barriers keep the pairs' operands from all being
            // built at once, which would not fit the registers)
#pragma unroll
            for (int r = 0; r < RG; r++) {
                if (p0 == 0) wr[r].settle();
                wr[r].hold();
                floatx4 t = KRK_ZERO4;
#define KRK_PAIR(P)                                                   \
    __builtin_amdgcn_sched_barrier(0);                                \
    wr[r].template pair<P>(xa[P], masks, t, acc[r]);                  \
    settle_acc(DT == DT_Q4_K || DT == DT_Q5_K ? t : acc[r]);          \
    if (r == RG - 1 && more) load_pair(P);                            \
    __builtin_amdgcn_sched_barrier(0);
                KRK_PAIR(0) KRK_PAIR(1) KRK_PAIR(2) KRK_PAIR(3)
#undef KRK_PAIR
                wr[r].finish(xs, masks, t, acc[r]);
                settle_acc(acc[r]);
                if (r == RG - 1 && more) load_sums();
            }
        }
        // lane (j, g): weight row j, activation rows 4g .. 4g + 3
#pragma unroll
        for (int r = 0; r < RG; r++)
#pragma unroll
            for (int k = 0; k < 4; k++) red[(wv * 16 + 4 * g + k) * S + 16 * r + j] = acc[r][k];
        __syncthreads();
        const int left = a.rows - p0 < per ? a.rows - p0 : per;
        for (int o = tid; o < left * rows_t; o += 64 * nw) {
            const int i = o >> rows_sh, c = o - (i << rows_sh), p = p0 + i;
            const int64_t n = n0 + c;
            if (n >= n_out) continue;
            // (requested before the sums, not after)
            const float inv = a.inv[p];
            const float v = wave_sums<NWMAX, NWX>(red + i * S + c, 16 * S, 8 * S, nw, a.planes);
            if (a.part) {   // this K range's partial
                __hip_atomic_store(a.part + blockIdx.z * prow + static_cast<int64_t>(p) * a.part_n +
                                       a.seg[blockIdx.y].col + n,
                                   v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                continue;
            }
            if (a.out_f16) static_cast<_Float16 *>(out)[p * n_out + n] = static_cast<_Float16>(v * inv);
            else static_cast<float *>(out)[p * n_out + n] = v * inv;
        }
        __syncthreads();
    }
    if (!a.part) return;
    // K ranges: each workgroup's partials are complete before it
    // counts itself in the tile's counter; the last to arrive adds the ranges'
    // partials in range order, so the result does not depend on which one
    // that is, and clears the counter for the next call.  Partials and
    // counter are agent-scope atomics: coherent across the XCDs' L2s without
    // a cache write-back or invalidate.
    __shared__ int is_last;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    unsigned *cnt = a.cnt + static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x;
    if (tid == 0)
        is_last = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.z - 1u;
    __syncthreads();
    if (!is_last) return;
    for (int o = tid; o < a.rows * rows_t; o += 64 * nw) {
        const int p = o >> rows_sh;
        const int64_t n = n0 + (o - (p << rows_sh));
        if (n >= n_out) continue;
        const float *src = a.part + static_cast<int64_t>(p) * a.part_n + a.seg[blockIdx.y].col + n;
        float v = 0.0f;
        for (unsigned z = 0; z < gridDim.z; z++)
            v += __hip_atomic_load(src + z * prow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        v *= a.inv[p];
        if (a.out_f16) static_cast<_Float16 *>(out)[p * n_out + n] = static_cast<_Float16>(v);
        else static_cast<float *>(out)[p * n_out + n] = v;
    }
    if (tid == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Routed.  Persistent workgroups over chunks of `ct` weight tiles of one active
// expert (chunk c: run c / chunks per run), its waves splitting K into slices
// of NBW blocks.  A tile is 16 RG weight rows (gate/up pairs: 8 RG gate rows
// and the same up rows), multiplied with the expert's prepared rows, 16 a pass.
// A row group's registers take the same group of the next tile as soon as its
// last pass is multiplied, and the activations stay in registers while the
// expert and its pass do (one-block slices), so the weights stream without a
// pause: one workgroup per tile with everything requested up front left the
// memory idle while it multiplied and summed (gate/up of 160 tokens, 906 MB:
// 339 -> 269 us, down, 453 MB: 189 -> 140 us; the loads alone take 3/4 of it).  The waves' sums alternate between two LDS buffers, one barrier a
// step; it is a bare one, so that the requests in flight stay so.
template <int DT, int NBW, int RG, int NWMAX, bool NWX>
__global__ void __launch_bounds__(64 * NWMAX) __attribute__((amdgpu_waves_per_eu(4)))
    rows_routed_kernel(RowsArgs a, int tiles, int ct) {
    extern __shared__ __align__(16) float red_lds[];
    constexpr int S = 16 * RG + 4;
    using At = PrepAt<false>;
    constexpr int H = RG / 2;               // row groups of each half of a pair
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = NWX ? NWMAX : static_cast<int>(blockDim.x) >> 6;
    const int j = lane & 15, g = lane >> 4;
    const int kb0 = wv * NBW;
    const int nbl = a.nb - kb0 < NBW ? a.nb - kb0 : NBW;    // blocks of this wave's slice (at least one)
    const bool pair = a.pair;
    const int rows_sh = (RG == 4 ? 6 : RG == 2 ? 5 : 4) - (pair ? 1 : 0), rows_t = 1 << rows_sh;
    const int per = a.planes == 2 ? 8 : 16;                 // rows a pass
    const int64_t n_out = a.seg[0].n_out;
    float *out = static_cast<float *>(a.seg[0].out);
    const int cpr = (tiles + ct - 1) / ct, chunks = *a.n_act * cpr;
    int chunk = static_cast<int>(blockIdx.x);
    if (chunk >= chunks) return;

    struct Step {
        const uint8_t *w, *w2;
        int tile, tend, pb, pe, p0;
    };
    auto open = [&](int c) {
        const int run = c / cpr;
        const EmRun &r = a.runs[run];
        Step s;
        s.w = static_cast<const uint8_t *>(r.w[pair ? 0 : 2]);
        s.w2 = static_cast<const uint8_t *>(r.w[1]);
        s.tile = (c - run * cpr) * ct;
        s.tend = s.tile + ct < tiles ? s.tile + ct : tiles;
        s.pb = s.p0 = r.pb;
        s.pe = r.pe;
        return s;
    };
    gbyte *xrow = nullptr;
    auto point = [&](const Step &s) {
        int p = s.p0 + (a.planes == 2 ? (j & 7) : j);
        p = p < s.pe ? p : s.p0;            // rows past the end re-read the pass's first
        const int64_t t = a.tok ? a.tok[p] : p;
        xrow = to_global(a.xp) + At::row(a.planes == 2 ? 2 * t + (j >> 3) : t, a.nb) +
               static_cast<int64_t>(kb0) * At::kBlock + At::kPiece * g;
    };
    u32x4 xa[4][2], xs = {0u, 0u, 0u, 0u};
    auto load_pair = [&](int p, int b) {
#pragma unroll
        for (int s = 0; s < 2; s++) xa[p][s] = ld128(xrow + b * At::kBlock + At::kPart * (2 * p + s));
    };
    auto load_sums = [&](int b) {
        if constexpr (has_min(DT)) xs = ld128(xrow + b * At::kBlock + At::kPart * 8);
    };
    const Masks masks;
    RowBlk<DT> wr[NBW][RG];
    // a uniform row base and a 32-bit lane offset (rows are shorter than 2^26
    // bytes); rows past the bank's last re-read it, a ragged last slice its
    // last block, unused
    const uint32_t rb = static_cast<uint32_t>(a.row_bytes);
    auto fetch = [&](const Step &s, int b, int r) {
        int64_t n = static_cast<int64_t>(s.tile) * rows_t + 16 * (pair && H && r >= H ? r - H : r);
        n = n < n_out ? n : n_out - 1;
        const int lim = n_out - n < 16 ? static_cast<int>(n_out - n) - 1 : 15;
        gbyte *base = to_global(pair && r >= H ? s.w2 : s.w) + n * a.row_bytes +
                      static_cast<int64_t>(kb0 + (b < nbl ? b : nbl - 1)) * RowBlk<DT>::BB;
        wr[b][r].fetch(base + static_cast<uint32_t>(j < lim ? j : lim) * rb, g);
    };
    Step cur = open(chunk);
    point(cur);
#pragma unroll
    for (int p = 0; p < 4; p++) load_pair(p, 0);
    load_sums(0);
#pragma unroll
    for (int b = 0; b < NBW; b++)
#pragma unroll
        for (int r = 0; r < RG; r++) fetch(cur, b, r);

    for (int buf = 0;; buf ^= 1) {
        // the next step: whether it brings another tile, other activations
        Step nxt = cur;
        bool wn = false, xn = true, end = false;
        if (cur.p0 + per < cur.pe) {
            nxt.p0 += per;
        } else {
            wn = true;
            nxt.p0 = cur.pb;
            if (++nxt.tile < cur.tend) {
                xn = cur.pe - cur.pb > per;
            } else {
                chunk += static_cast<int>(gridDim.x);
                end = chunk >= chunks;
                if (!end) nxt = open(chunk);
                wn = xn = !end;
            }
        }
        const bool xr = !end && (xn || nbl > 1);
        // this thread's first output's row scale, needed after the barrier
        const int left = cur.pe - cur.p0 < per ? cur.pe - cur.p0 : per;
        const int i0 = tid >> rows_sh;
        const int t0 = i0 < left ? cur.p0 + i0 : cur.p0;
        float inv = a.inv[a.tok ? a.tok[t0] : t0];
        floatx4 acc[RG];
#pragma unroll
        for (int r = 0; r < RG; r++) acc[r] = KRK_ZERO4;
#pragma unroll
        for (int b = 0; b < NBW; b++) {
            if (b >= nbl) break;            // wave-uniform
            const bool last = b + 1 >= nbl, refill = !last || xr;
            const int nb = last ? 0 : b + 1;
            if (last && xr) point(nxt);
#pragma unroll
            for (int r = 0; r < RG; r++) {
                if (cur.p0 == cur.pb) wr[b][r].settle();
                wr[b][r].hold();
                floatx4 t = KRK_ZERO4;
#define KRK_PAIR(P)                                                   \
    __builtin_amdgcn_sched_barrier(0);                                \
    wr[b][r].template pair<P>(xa[P], masks, t, acc[r]);               \
    settle_acc(DT == DT_Q4_K || DT == DT_Q5_K ? t : acc[r]);          \
    if (r == RG - 1 && refill) load_pair(P, nb);                      \
    __builtin_amdgcn_sched_barrier(0);
                KRK_PAIR(0) KRK_PAIR(1) KRK_PAIR(2) KRK_PAIR(3)
#undef KRK_PAIR
                wr[b][r].finish(xs, masks, t, acc[r]);
                settle_acc(acc[r]);
                if (r == RG - 1 && refill) load_sums(nb);
                if (wn) fetch(nxt, b, r);
            }
        }
        float *red = red_lds + buf * (nw * 16 * S);
#pragma unroll
        for (int r = 0; r < RG; r++)
#pragma unroll
            for (int k = 0; k < 4; k++) red[(wv * 16 + 4 * g + k) * S + 16 * r + j] = acc[r][k];
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const int64_t n0 = static_cast<int64_t>(cur.tile) * rows_t;
        for (int o = tid; o < left * rows_t; o += 64 * nw) {
            const int i = o >> rows_sh, c = o - (i << rows_sh), p = cur.p0 + i;
            const int64_t n = n0 + c;
            if (o != tid) inv = a.inv[a.tok ? a.tok[p] : p];
            if (n >= n_out) continue;
            float v = wave_sums<NWMAX, NWX>(red + i * S + c, 16 * S, 8 * S, nw, a.planes) * inv;
            if (pair) {
                float up = wave_sums<NWMAX, NWX>(red + i * S + 16 * H + c, 16 * S, 8 * S, nw, a.planes) * inv;
                if (a.act_f16) {
                    // both dots rounded to f16 first, silu with the device
                    // exponential (moe_table.hpp:250-253)
                    v = static_cast<float>(static_cast<_Float16>(v));
                    up = static_cast<float>(static_cast<_Float16>(up));
                    v = silu_f(v) * up;
                } else {
                    v = (v / (1.0f + expf(-v))) * up;
                }
            }
            out[p * n_out + n] = v;
        }
        if (end) break;
        cur = nxt;
    }
}

template <int DT, int RG> hipError_t launch(const RowsArgs &a, dim3 grid, int nw, hipStream_t st) {
    const size_t lds = static_cast<size_t>(nw) * 16 * (16 * RG + 4) * sizeof(float);
    if (nw == 8)
        hipLaunchKernelGGL((rows_kernel<DT, RG, 8, true>), grid, dim3(64 * nw), lds, st, a);
    else if (nw < 8)
        hipLaunchKernelGGL((rows_kernel<DT, RG, 8, false>), grid, dim3(64 * nw), lds, st, a);
    else if (nw == kRowsWaves)
        hipLaunchKernelGGL((rows_kernel<DT, RG, kRowsWaves, true>), grid, dim3(64 * nw), lds, st, a);
    else
        hipLaunchKernelGGL((rows_kernel<DT, RG, kRowsWaves, false>), grid, dim3(64 * nw), lds, st, a);
    return hipGetLastError();
}

template <int DT, int NBW, int RG>
hipError_t launch_routed(const RowsArgs &a, int nw, hipStream_t st) {
    const size_t lds = static_cast<size_t>(2) * nw * 16 * (16 * RG + 4) * sizeof(float);
    const int64_t rows_t = 16 * (a.pair ? RG / 2 : RG);
    if (rows_t < 1 || a.max_runs < 1) return hipErrorNotSupported;
    const int64_t tiles = (a.seg[0].n_out + rows_t - 1) / rows_t;
    if (tiles * a.max_runs >= (int64_t{1} << 31)) return hipErrorNotSupported;
    // as many workgroups as are resident (the registers allow sixteen waves a
    // compute unit), chunks of up to eight tiles while every one gets four
    const int64_t wgs = static_cast<int64_t>(device_cus()) * (nw <= 4 ? 4 : nw <= 5 ? 3 : nw <= 8 ? 2 : 1);
    int64_t ct = tiles * a.max_runs / (4 * wgs);
    ct = ct < 1 ? 1 : ct > 8 ? 8 : ct;
    const int64_t chunks = (tiles + ct - 1) / ct * a.max_runs;
    const dim3 grid(static_cast<unsigned>(chunks < wgs ? chunks : wgs));
    const int t = static_cast<int>(tiles), c = static_cast<int>(ct);
    if (nw == 8)
        hipLaunchKernelGGL((rows_routed_kernel<DT, NBW, RG, 8, true>), grid, dim3(64 * nw), lds, st, a, t, c);
    else if (nw < 8)
        hipLaunchKernelGGL((rows_routed_kernel<DT, NBW, RG, 8, false>), grid, dim3(64 * nw), lds, st, a, t, c);
    else if (nw == kRowsWaves)
        hipLaunchKernelGGL((rows_routed_kernel<DT, NBW, RG, kRowsWaves, true>), grid, dim3(64 * nw), lds, st, a, t, c);
    else
        hipLaunchKernelGGL((rows_routed_kernel<DT, NBW, RG, kRowsWaves, false>), grid, dim3(64 * nw), lds, st, a, t, c);
    return hipGetLastError();
}

// The tiling of a launch: row groups and blocks per wave, K ranges and their
// blocks, waves.
struct RowsShape {
    int nbw, rg, range, splits, nw;
};
RowsShape rows_shape(const RowsArgs &a, int dt, int nb) {   // (reads runs, n and the segments' n_out)
    RowsShape s{};
    // (Q6_K's and Q8_0's blocks of four row groups do not fit the registers)
    const bool wide = dt != DT_Q8_0 && dt != DT_Q6_K;
    if (a.runs) {
        s.nbw = (nb + kRowsWaves - 1) / kRowsWaves;
        s.rg = s.nbw == 1 ? (wide ? 4 : 2) : s.nbw == 2 ? 2 : 1;
        s.splits = 1;
        s.range = nb;
    } else {
        // dense: one block a wave and K ranges of at most 16 blocks
        int64_t n = 0;
        for (int i = 0; i < a.n; i++) n += a.seg[i].n_out;
        s.nbw = 1;
        s.splits = (nb + kRowsWaves - 1) / kRowsWaves;
        s.range = (nb + s.splits - 1) / s.splits;
        const int64_t cus = device_cus();
        s.rg = wide && (n + 63) / 64 * s.splits >= cus * 3 / 4 ? 4 : (n + 31) / 32 * s.splits >= cus * 3 / 4 ? 2 : 1;
    }
    s.nw = (s.range + s.nbw - 1) / s.nbw;
    return s;
}

template <int DT> hipError_t launch_shape(const RowsArgs &a, const RowsShape &s, hipStream_t st) {
    constexpr bool WIDE = DT != DT_Q8_0 && DT != DT_Q6_K;
    if (a.runs) {
        switch (s.nbw) {
            case 1: return launch_routed<DT, 1, WIDE ? 4 : 2>(a, s.nw, st);
            case 2: return launch_routed<DT, 2, 2>(a, s.nw, st);
            case 3: return launch_routed<DT, 3, 1>(a, s.nw, st);
            case 4: return launch_routed<DT, 4, 1>(a, s.nw, st);
            default: return hipErrorNotSupported;
        }
    }
    int64_t widest = 0;
    for (int i = 0; i < a.n; i++) widest = a.seg[i].n_out > widest ? a.seg[i].n_out : widest;
    const int64_t width = (widest + 16 * s.rg - 1) / (16 * s.rg);
    if (width >= (int64_t{1} << 31) || (s.splits > 1 && (!a.part || width * a.n > kTileCounters)))
        return hipErrorNotSupported;
    const dim3 grid(static_cast<unsigned>(width), static_cast<unsigned>(a.n), static_cast<unsigned>(s.splits));
    if constexpr (WIDE)
        if (s.rg == 4) return launch<DT, 4>(a, grid, s.nw, st);
    return s.rg == 2 ? launch<DT, 2>(a, grid, s.nw, st) : launch<DT, 1>(a, grid, s.nw, st);
}

}  // namespace

bool gemm_rows_tiles_ok(int dt, int64_t n_in, const int64_t n_out[], int n, bool counters) {
    RowsArgs a{};
    if (n < 1 || n > kMaxSegs) return false;
    int64_t widest = 0;
    for (int i = 0; i < n; i++) {
        a.seg[i].n_out = n_out[i];
        widest = n_out[i] > widest ? n_out[i] : widest;
    }
    a.n = n;
    const RowsShape s = rows_shape(a, dt, static_cast<int>(n_in / 256));
    return s.splits == 1 || (counters && (widest + 16 * s.rg - 1) / (16 * s.rg) * n <= kTileCounters);
}

bool gemm_rows_ok(int dt, int64_t n_in, const void *w, int64_t row_bytes) {
    switch (dt) {
        case DT_Q4_K: case DT_Q5_K:
            if ((reinterpret_cast<uintptr_t>(w) | static_cast<uintptr_t>(row_bytes)) & 15) return false;
            break;
        case DT_Q6_K: case DT_Q8_0: case DT_Q4_0:
            if ((reinterpret_cast<uintptr_t>(w) | static_cast<uintptr_t>(row_bytes)) & 1) return false;
            break;
        default: return false;
    }
    return n_in > 0 && n_in % 256 == 0 && n_in / 256 <= kRowsWaves * kRowsBlocks;   // (rows well under 2^26 bytes)
}

static size_t prep_rows_bytes(int64_t rows, int64_t n_in, int planes, bool dense) {
    const int nb = static_cast<int>(n_in / 256);
    const int64_t r = rows * planes;
    const int64_t n = dense ? (r + 15) / 16 * PrepAt<true>::stride(nb) : r * PrepAt<false>::stride(nb);
    return (static_cast<size_t>(n) + 255) & ~size_t(255);
}

size_t gemm_rows_prep_bytes(int64_t rows, int64_t n_in, int planes, bool dense) {
    return prep_rows_bytes(rows, n_in, planes, dense) + ((rows * sizeof(float) + 255) & ~size_t(255));
}

size_t gemm_rows_part_bytes(int64_t rows, int64_t n_total, int64_t n_in) {
    const int64_t splits = (n_in / 256 + kRowsWaves - 1) / kRowsWaves;
    return splits > 1 ? static_cast<size_t>(splits) * rows * n_total * sizeof(float) : 0;
}

hipError_t gemm_rows_prep(int dt, const void *x, bool x_f16, int64_t x_stride, int64_t rows, int64_t n_in, int planes,
                          bool dense, const int32_t *n_rows, void *ws, RowsArgs &a, hipStream_t st) {
    if (rows < 1 || rows >= (int64_t{1} << 31) || n_in % 256 || (reinterpret_cast<uintptr_t>(x) & 15) || x_stride % 8)
        return hipErrorInvalidValue;
    const int nb = static_cast<int>(n_in / 256);
    uint8_t *xp = static_cast<uint8_t *>(ws);
    float *inv = reinterpret_cast<float *>(xp + prep_rows_bytes(rows, n_in, planes, dense));
    const dim3 grid(static_cast<unsigned>(rows), static_cast<unsigned>((nb + 31) / 32));
#define KRK_PREP_AS(D, T, DENSE)                                                                             \
    hipLaunchKernelGGL((rows_prep_kernel<D, T, DENSE>), grid, dim3(256), 0, st, static_cast<const T *>(x), x_stride, \
                       nb, planes, n_rows, xp, inv)
#define KRK_PREP(D)                                                                                          \
    case D:                                                                                                  \
        if (x_f16 && dense) KRK_PREP_AS(D, _Float16, true);                                                  \
        else if (x_f16) KRK_PREP_AS(D, _Float16, false);                                                     \
        else if (dense) KRK_PREP_AS(D, float, true);                                                         \
        else KRK_PREP_AS(D, float, false);                                                                   \
        break;
    switch (dt) {
        KRK_PREP(DT_Q4_K) KRK_PREP(DT_Q5_K) KRK_PREP(DT_Q6_K) KRK_PREP(DT_Q8_0) KRK_PREP(DT_Q4_0)
        default: return hipErrorNotSupported;
    }
#undef KRK_PREP
#undef KRK_PREP_AS
    a.xp = xp;
    a.inv = inv;
    a.planes = planes;
    a.nb = nb;
    return hipGetLastError();
}

hipError_t gemm_rows(int dt, const RowsArgs &a0, hipStream_t st) {
    RowsArgs a = a0;
    if (a.nb < 1 || a.nb > kRowsWaves * kRowsBlocks || (a.pair && (a.nb > 32 || !a.runs)) ||
        (!a.runs && (a.n < 1 || a.n > kMaxSegs)))
        return hipErrorNotSupported;
    const RowsShape s = rows_shape(a, dt, a.nb);
    a.range = s.range;
    if (s.splits == 1) a.part = nullptr;
    else if (!a.part || !a.cnt) return hipErrorNotSupported;
    a.part_n = 0;
    for (int i = 0; i < a.n; i++) {
        a.seg[i].col = a.part_n;
        a.part_n += a.seg[i].n_out;
    }
    switch (dt) {
#define KRK_ROWS(D) \
    case D: return launch_shape<D>(a, s, st);
        KRK_ROWS(DT_Q4_K) KRK_ROWS(DT_Q5_K) KRK_ROWS(DT_Q6_K) KRK_ROWS(DT_Q8_0) KRK_ROWS(DT_Q4_0)
#undef KRK_ROWS
        default: return hipErrorNotSupported;
    }
}

}  // namespace krk
