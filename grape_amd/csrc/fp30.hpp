// Fp on signed limbs of 30 bits with lazy reduction - the working form of the commitment kernels
// (13 limbs, radix 2^390, for BLS12-381; 9 limbs, radix 2^270, for BN254).
//
// Why: on gfx950 a 32x32+64 multiply-add (v_mad_i64_i32 / v_mad_u64_u32) issues at the same rate
// as an addition, so the cost of a field product is its instruction count, and with saturated
// 32-bit limbs two thirds of the instructions are carry handling.  Signed limbs make subtraction
// limb-wise, and BALANCED ones - digits in [-2^29, 2^29) - have products below 2^58, so that a whole
// column of an (a*b + m*p) row set fits a signed 64-bit accumulator with limbs of 30 bits: 13 limbs where
// unsigned digits need 28 bits and 14 limbs (338 instead of 392 multiply-adds a product).
//
// Representation: x = sum_i v[i] * 2^(30 i), v[i] signed 32-bit.  "Balanced": |v[i]| <= 2^29 + 2 for
// i < N-1, the top limb carries what is left.  "Normalised": 0 <= v[i] < 2^30 for i < N-1, the top
// limb carries the sign - the form in which values are compared.  A value stands for its residue mod p;
// arithmetic is Montgomery with radix R' = 2^(30 N).  The canonical memory form elsewhere in the
// library is the reference's: 32-bit limbs, radix 2^384 resp. 2^256 (include/field/mont_t.cuh,
// include/field/bls12-381.cuh:7-23, include/field/alt_bn128.cuh); conversion is exact both ways.
//
// Reduction: T = T0 + 2^30 T1 becomes T1 + T0 * (2^-30 mod p), column by column - the quotient digit
// is the column's low 30 bits as they stand, with no product to find it and no carry to wait
// for.  The factor 2^-30 mod p is taken nearest to zero (for BLS12-381 2^369: p^-1 mod 2^30
// has 18 bits).  With balanced operands the columns have room for digits of 32 bits, whose cut is a column's word
// boundary.  The last column takes the ordinary step (a digit of -T0/p, times p), so that the result does not
// carry the factor 2^30 that the others would leave in it.
//
// Bounds (checked by the callers' comments).  Values: mul30(a, b) with |a| < alpha*p, |b| < beta*p
// is a balanced number of magnitude below (0.51 + alpha*beta/630) p; for BN254 0.94 p (1.4 p from wide digits)
// instead of 0.51 p, and 86000 instead of 630 - below p for every product here, wide digits on BN254 apart, so that a
// product is zero mod p only when all its limbs are zero.  Columns: a sum of 12 limb products of balanced operands is
// 0.38 * 2^63, the reduction adds 0.24 (0.48 in wide digits); so ONE operand may be a lazy sum or difference of two balanced numbers or
// normalised (0.985 * 2^63 in the worst column; BN254 0.77), and so may two products of balanced operands share
// their columns.  Lazy operands on both sides do not fit: balance() one.
#pragma once
#include "curve.hpp"
#include "divstep.hpp"

namespace grape {

#if defined(GRAPE_CURVE_BN254)
struct Fp30 {
    int32_t v[9];
};

namespace fp30 {

using detail::mad;
using detail::unknown;

constexpr int N = 9;
constexpr int W = 30;
constexpr bool kSmallDown = false;
constexpr uint32_t PINV = 0x24866389u;   // -p^-1 mod 2^30

GRAPE_HD int32_t P(int i) {   // balanced, as all tables of limbs here
    constexpr int32_t t[9] = {0x187cfd47, -0xf7dcfa5, 0x71ca8d4, -0x1fa55ba6, 0x1585d98, 0x116da06, 0x1a029b85, 0x139cb84c, 0x3064};
    return t[i];
}
GRAPE_HD int32_t P2(int i) {   // 2p
    constexpr int32_t t[9] = {-0xf060572, -0x1efb9f49, 0xe3951a8, 0xb548b4, 0x2b0bb2f, 0x22db40c, -0xbfac8f6, -0x18c68f67, 0x60c9};
    return t[i];
}
GRAPE_HD int32_t P3(int i) {   // 3p
    constexpr int32_t t[9] = {0x976f7d5, 0x11869112, 0x1555fa7b, -0x1ef012f2, 0x40918c7, 0x3448e12, 0xe07d28f, -0x529d71b, 0x912d};
    return t[i];
}
GRAPE_HD int32_t DOWN(int i) {   // 2^-30 mod p: -0.43 p
    constexpr int32_t t[9] = {0x1f7dceac, 0x193ed8c9, 0xa1f275e, 0xfa1c301, -0x1de4d6a1, 0x8aff355, -0x93e8175, -0x1142d07b, -0x14c6};
    return t[i];
}
GRAPE_HD int32_t ONE(int i) {   // 2^270 mod p
    constexpr int32_t t[9] = {0x24fcf82, -0xe183b72, 0x1ac0210c, 0x1f4f4b0c, 0x100896b9, -0xae44a8a, -0x6d2519d, -0x1ab5fcf1, -0x8c8};
    return t[i];
}
GRAPE_HD int32_t CMEM(int i) {   // 2^256 mod p: mul30(x*2^270, CMEM) = x*2^256
    constexpr int32_t t[9] = {0x58f0d9d, 0xd750e37, 0x1c70b3dd, 0x1e3aca3d, -0x6b9d3f6, -0x572421e, -0x20d0999, 0x1df06682, 0xe0a};
    return t[i];
}
// Montgomery (radix 2^256) form of 2^14, 32-bit limbs: mul(x*2^256, MCONV) = x*2^270 mod p
GRAPE_HD uint32_t MCONV(int i) {
    constexpr uint32_t t[8] = {0x5accccc9u, 0xf89a7d3au, 0x9a1dcc9du, 0x50fea7bdu, 0xdf1160f4u, 0x9e7d8ca3u, 0xed6d3304u, 0x279be39au};
    return t[i];
}
GRAPE_HD int32_t CIN(int i) {   // 2^284 mod p: mul30(pack(x*2^256), CIN) = x*2^270
    constexpr int32_t t[9] = {-0x1019212e, -0x66eb814, -0x18cbc210, -0x103b9669, 0x63da561, 0x14d661fb, 0x15e36864, 0x1768c0ce, 0x1291};
    return t[i];
}
GRAPE_HD int32_t R3(int i) {   // R'^3 mod p: turns the plain inverse of a Montgomery-form value back into Montgomery form
    constexpr int32_t t[9] = {0x70aee79, 0x85cef6a, -0x17012488, 0x1859261c, 0x1a5cb6c3, -0x495f3be, 0x179e76b2, 0x17c5ea5a, 0x574};
    return t[i];
}

#else
struct Fp30 {
    int32_t v[13];
};

namespace fp30 {

using detail::mad;
using detail::unknown;

constexpr int N = 13;
constexpr int W = 30;
constexpr bool kSmallDown = true;        // DOWN is far below p
constexpr uint32_t PINV = 0x3ffcfffdu;   // -p^-1 mod 2^30

GRAPE_HD int32_t P(int i) {   // balanced, as all tables of limbs here
    constexpr int32_t t[13] = {-0x5555, -0x18040000, 0x153ffffc, -0x15000054, -0xf09dbe1, 0x34a83db, 0x112bf673,
                               0x12e13ce1, -0x13289b89, 0x1ed90d2f, -0x165b4e46, -0x571a006, 0x1a0112};
    return t[i];
}
GRAPE_HD int32_t P2(int i) {   // 2p
    constexpr int32_t t[13] = {-0xaaaa, 0xff80000, -0x15800009, 0x15ffff59, -0x1e13b7c3, 0x69507b6, -0x1da8131a,
                               -0x1a3d863d, 0x19aec8ef, -0x24de5a3, 0x13496375, -0xae3400d, 0x340224};
    return t[i];
}
GRAPE_HD int32_t P3(int i) {   // 3p
    constexpr int32_t t[13] = {-0xffff, -0x80c0000, -0x40000d, 0xffff05, 0x12e26c5c, 0x9df8b90, -0xc7c1ca7,
                               -0x75c495c, 0x6862d66, 0x1c8b278c, -0x311ead1, -0x1054e013, 0x4e0336};
    return t[i];
}
GRAPE_HD int32_t DOWN(int i) {   // 2^-30 mod p: -0.0002 p
    constexpr int32_t t[13] = {0x80c0004, 0x4d203d, -0x4fe05, 0xc18fa4, -0x156fd71a, -0x16dd0ad7, 0x10b87b4d,
                               0xc13f00b, -0x41741a5, -0x121d875c, -0xf9813a5, -0x383c1e2, -0x138};
    return t[i];
}
GRAPE_HD int32_t ONE(int i) {   // 2^390 mod p
    constexpr int32_t t[13] = {0xd1ff2e, 0x19d80000, -0xb7ff53c, -0x11ff3219, 0x2431c85, -0x19607c5e, -0x2307f22,
                               0x9b42da1, -0x1a113d94, 0x15d98f13, 0x4b29f14, -0x1a603060, 0x15dea};
    return t[i];
}
GRAPE_HD int32_t CMEM(int i) {   // 2^384 mod p: mul30(x*2^390, CMEM) = x*2^384
    constexpr int32_t t[13] = {0x35552, -0xfd80000, -0x147fffd4, 0x12000345, 0x166296cd, 0x1f16d974, 0x14485f81,
                               0x3339f33, -0x69eca9, 0xb857c2d, 0x1f910eb7, -0x98fbfc1, -0x40ab3};
    return t[i];
}
// Montgomery (radix 2^384) form of 2^6, 32-bit limbs: mul(x*2^384, MCONV) = x*2^390 mod p
GRAPE_HD uint32_t MCONV(int i) {
    constexpr uint32_t t[12] = {0x00d1ff2eu, 0x46760000u, 0x9b4800acu, 0x84b80337u, 0xe882431cu, 0x0dd9a7e0u,
                                0xb683dcf8u, 0xc26c26d0u, 0x63c4a5eeu, 0x29f14576u, 0x7f3e804bu, 0x015de996u};
    return t[i];
}
GRAPE_HD int32_t CIN(int i) {   // 2^396 mod p: mul30(pack(x*2^384), CIN) = x*2^390
    constexpr int32_t t[13] = {-0xb7f3481, -0x1f3ffff, -0x1fbd4ed9, -0xcc8550, -0x21b4b2e, 0x1e015cf2, 0x5c540d,
                               -0xb984e66, -0xad5925c, 0x19d89d1a, -0x1046501a, -0x7b737e8, 0x97730};
    return t[i];
}
GRAPE_HD int32_t R3(int i) {   // R'^3 mod p: turns the plain inverse of a Montgomery-form value back into Montgomery form
    constexpr int32_t t[13] = {0x1347c98d, -0x13de6b34, 0x1b027ceb, -0x14734a5b, 0x1214bbdf, 0xb5efd04, -0x6122f41,
                               0x1b2b39a5, -0xd4ff49a, 0x1d1b6db5, -0x470f471, 0x12c853b8, 0x6d0af};
    return t[i];
}

#endif

constexpr uint32_t MASK = (1u << W) - 1;
constexpr int32_t HALF = 1 << (W - 1);

GRAPE_HD Fp30 one() {
    Fp30 r;
#pragma unroll
    for (int i = 0; i < N; i++) r.v[i] = ONE(i);
    return r;
}
GRAPE_HD Fp30 zero() {
    Fp30 r;
#pragma unroll
    for (int i = 0; i < N; i++) r.v[i] = 0;
    return r;
}

// limb-wise, no carries: the caller tracks magnitudes
GRAPE_HD Fp30 sub(const Fp30& a, const Fp30& b) {
    Fp30 r;
#pragma unroll
    for (int i = 0; i < N; i++) r.v[i] = a.v[i] - b.v[i];
    return r;
}
GRAPE_HD Fp30 cneg(const Fp30& a, bool flag) {
    Fp30 r;
    const int32_t m = flag ? -1 : 0;
#pragma unroll
    for (int i = 0; i < N; i++) r.v[i] = (a.v[i] ^ m) - m;
    return r;
}

// signed carry propagation: same value, limbs 0..N-2 in [0, 2^30); any 32-bit limbs
GRAPE_HD Fp30 normalize(const Fp30& a) {
    Fp30 r;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < N - 1; i++) {
        const int32_t t = (int32_t)((uint32_t)a.v[i] & MASK) + c;
        r.v[i] = (int32_t)((uint32_t)t & MASK);
        c = (a.v[i] >> W) + (t >> W);   // arithmetic
    }
    r.v[N - 1] = a.v[N - 1] + c;
    return r;
}
GRAPE_HD int32_t low30(uint32_t a) { return (int32_t)(a << (32 - W)) >> (32 - W); }   // the nearest to zero of a's residues mod 2^30
// same value, balanced (up to 2 over 2^29: the limbs' carries are taken side by side, not along a chain).  Limbs below
// 3 * 2^29 - a sum or difference of two balanced numbers, a double - or, with ANY, any of 32 bits.
template <bool ANY = false>
GRAPE_HD Fp30 balance(const Fp30& a) {
    Fp30 r;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < N - 1; i++) {
        r.v[i] = low30((uint32_t)a.v[i]) + c;
        c = ANY ? ((a.v[i] >> (W - 1)) + 1) >> 1 : (a.v[i] + HALF) >> W;
    }
    r.v[N - 1] = a.v[N - 1] + c;
    return r;
}

// The columns of a double-width value, column k of weight 2^(30 k).  The upper ones hold 2^29 more than their value
// from the start, so that cutting their low 30 bits off rounds to the nearest multiple of 2^30; with WIDE, the lower
// ones 2^31 more, so that their upper word is the nearest multiple of 2^32.
struct Columns {
    int64_t c[2 * N - 1];
};
template <bool WIDE>
GRAPE_HD void start(Columns& t) {
    const int64_t lower = WIDE ? unknown((int64_t)1 << 31) : 0, upper = unknown((int64_t)HALF);
#pragma unroll
    for (int k = 0; k < 2 * N - 1; k++) t.c[k] = k < N - 1 ? lower : k < N ? 0 : upper;
}
GRAPE_HD void add_row(Columns& t, int i, const int32_t* a, int32_t b) {
#pragma unroll
    for (int j = 0; j < N; j++) mad(t.c[i + j], a[j], b);
}
// takes column i, which nothing is added to any more, out of the value
template <bool WIDE>
GRAPE_HD void reduce_column(Columns& t, int i) {
    if (i < N - 1) {
        int32_t m;
        if (WIDE) {                      // a signed digit of 32 bits: one instruction less for the column's upper part
            m = (int32_t)((uint32_t)t.c[i] ^ 0x80000000u);
            mad(t.c[i + 1], (int32_t)(t.c[i] >> 32), unknown(4));
        } else {
            m = (int32_t)((uint32_t)t.c[i] & MASK);
            t.c[i + 1] += t.c[i] >> W;
        }
#pragma unroll
        for (int j = 0; j < N; j++) mad(t.c[i + 1 + j], m, DOWN(j));
    } else {
        const int32_t m = low30((uint32_t)t.c[i] * PINV);
#pragma unroll
        for (int j = 0; j < N; j++) mad(t.c[i + j], m, P(j));
        t.c[i + 1] += t.c[i] >> W;       // the column is a multiple of 2^30 now
    }
}
// the upper columns, carries propagated: the upper words along the columns, the two bits left over above a limb's 30 to the next limb
GRAPE_HD Fp30 finish(Columns& t) {
    Fp30 r;
    int32_t over = 0;
#pragma unroll
    for (int k = 0; k < N - 1; k++) {
        const uint32_t lo = (uint32_t)t.c[N + k];
        const int32_t hi = (int32_t)(t.c[N + k] >> 32);
        if (k < N - 2) mad(t.c[N + k + 1], hi, unknown(4));
        r.v[k] = (int32_t)(lo & MASK) + over - HALF;
        over = (int32_t)(lo >> W);
        if (k == N - 2) r.v[N - 1] = (int32_t)((uint32_t)hi << 2) + over;
    }
    return r;
}
// the same less w * s: an addend costs a multiply-add a limb here, and the difference comes out balanced
GRAPE_HD void less(Columns& t, int32_t& top, const Fp30& s, int32_t w) {
    const int32_t f = unknown(-w);
#pragma unroll
    for (int k = 0; k < N - 1; k++) mad(t.c[N + k], s.v[k], f);
    top += s.v[N - 1] * f;
}

// Montgomery product a*b/R' (mod p)
template <bool WIDE>
GRAPE_HD Fp30 mul_impl(const Fp30& a, const Fp30& b) {
    Columns t;
    start<WIDE>(t);
#pragma unroll
    for (int i = 0; i < N; i++) {
        add_row(t, i, a.v, b.v[i]);
        reduce_column<WIDE>(t, i);
    }
    return finish(t);
}
GRAPE_HD Fp30 mul(const Fp30& a, const Fp30& b) { return mul_impl<false>(a, b); }
// both operands balanced: reduced in wide digits, 12 instructions less
GRAPE_HD Fp30 mulb(const Fp30& a, const Fp30& b) { return mul_impl<true>(a, b); }
// both operands balanced, the product below p (wide digits take DOWN twice: too much where that is near p / 2)
GRAPE_HD Fp30 mulb_below_p(const Fp30& a, const Fp30& b) { return mul_impl<kSmallDown>(a, b); }
// a*b/R' - s, both factors balanced
GRAPE_HD Fp30 mulb_less(const Fp30& a, const Fp30& b, const Fp30& s) {
    Columns t;
    start<true>(t);
    int32_t top = 0;
    less(t, top, s, 1);
#pragma unroll
    for (int i = 0; i < N; i++) {
        add_row(t, i, a.v, b.v[i]);
        reduce_column<true>(t, i);
    }
    Fp30 r = finish(t);
    r.v[N - 1] += top;
    return r;
}

// a*b - c*d with one Montgomery reduction: both products accumulate in the same columns, so all four operands have to be
// balanced.
GRAPE_HD Fp30 mul_sub(const Fp30& a, const Fp30& b, const Fp30& c, const Fp30& d) {
    Columns t;
    start<false>(t);
    int32_t nc[N];                        // limb-wise negation keeps every step a multiply-add
#pragma unroll
    for (int j = 0; j < N; j++) nc[j] = -c.v[j];
#pragma unroll
    for (int i = 0; i < N; i++) {
        add_row(t, i, a.v, b.v[i]);
        add_row(t, i, nc, d.v[i]);
        reduce_column<false>(t, i);
    }
    return finish(t);
}

// the columns of a^2 (a balanced): the off-diagonal limb products are taken once with a doubled operand
template <bool WIDE>
GRAPE_HD void square(Columns& t, const Fp30& a) {
    int32_t a2[N];
#pragma unroll
    for (int i = 0; i < N; i++) a2[i] = a.v[i] * 2;
#pragma unroll
    for (int i = 0; i < N; i++) {
        mad(t.c[2 * i], a.v[i], a.v[i]);
#pragma unroll
        for (int j = i + 1; j < N; j++) mad(t.c[i + j], a2[i], a.v[j]);
    }
#pragma unroll
    for (int i = 0; i < N; i++) reduce_column<WIDE>(t, i);
}
template <bool WIDE>
GRAPE_HD Fp30 sqr_impl(const Fp30& a) {
    Columns t;
    start<WIDE>(t);
    square<WIDE>(t, a);
    return finish(t);
}
GRAPE_HD Fp30 sqr(const Fp30& a) { return sqr_impl<true>(a); }
GRAPE_HD Fp30 sqr_below_p(const Fp30& a) { return sqr_impl<kSmallDown>(a); }
// a^2/R' - s - 2u
GRAPE_HD Fp30 sqr_less(const Fp30& a, const Fp30& s, const Fp30& u) {
    Columns t;
    start<true>(t);
    int32_t top = 0;
    less(t, top, s, 1);
    less(t, top, u, 2);
    square<true>(t, a);
    Fp30 r = finish(t);
    r.v[N - 1] += top;
    return r;
}

// Is a product below p congruent to zero?
GRAPE_HD bool is_zero(const Fp30& a) {
    uint32_t z = 0;
#pragma unroll
    for (int i = 0; i < N; i++) z |= (uint32_t)a.v[i];
    return z == 0;
}
// Is a value of up to a few p, one lazy operand, congruent to zero?
GRAPE_HD bool is_zero_mod_p(const Fp30& a) { return is_zero(mul(a, one())); }

// the value in [0, p), normalised, of a product below p
GRAPE_HD Fp30 canonical(const Fp30& product) {
    Fp30 t = normalize(product);
    const int32_t neg = t.v[N - 1] >> 31;
#pragma unroll
    for (int i = 0; i < N; i++) t.v[i] += P(i) & neg;
    return normalize(t);
}

// ---- conversions with the canonical 32-bit-limb Montgomery form (radix 2^384 resp. 2^256) ----
constexpr int FW = FpParams::N;   // 32-bit words of the canonical form
// pure re-limbing of a non-negative integer of FW words (normalised)
GRAPE_HD Fp30 pack(const Fp& x) {
    Fp30 r;
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int bit = W * k, q = bit >> 5, s = bit & 31;
        uint64_t two = (uint64_t)x.v[q] | ((q + 1 < FW) ? ((uint64_t)x.v[q + 1] << 32) : 0);
        r.v[k] = (int32_t)((uint32_t)(two >> s) & MASK);
    }
    return r;
}
// inverse of pack for a normalised, non-negative value below 2^(32 FW)
GRAPE_HD Fp unpack(const Fp30& a) {
    Fp r;
#pragma unroll
    for (int q = 0; q < FW; q++) {
        // word q covers bits [32q, 32q+32): limbs k0 = floor(32q/30) .. up to two more
        const int k0 = (32 * q) / W;
        uint64_t acc = 0;
#pragma unroll
        for (int t = 0; t < 3; t++) {
            const int k = k0 + t;
            if (k < N) {
                const int sh = W * k - 32 * q;   // position of limb k relative to the word
                if (sh >= 0) {
                    if (sh < 32) acc |= (uint64_t)(uint32_t)a.v[k] << sh;
                } else {
                    acc |= (uint64_t)(uint32_t)a.v[k] >> (-sh);
                }
            }
        }
        r.v[q] = (uint32_t)acc;
    }
    return r;
}
// canonical memory form (32-bit limbs) -> the value in [0, p) in the working form, balanced
GRAPE_HD Fp30 from_canonical(const Fp& x) {
    Fp m;
#pragma unroll
    for (int i = 0; i < FW; i++) m.v[i] = MCONV(i);
    return balance(pack(fmul(x, m)));
}
// the same conversion with the 30-bit multiplier only (a third of the instructions): a product, so in
// (-p, p) instead of canonical
GRAPE_HD Fp30 from_canonical_lazy(const Fp& x) {
    Fp30 c;
#pragma unroll
    for (int i = 0; i < N; i++) c.v[i] = CIN(i);
    return mul(pack(x), c);
}
// value of up to a few p, one lazy operand -> canonical memory form, 32-bit limbs
GRAPE_HD Fp to_canonical(const Fp30& a) {
    Fp30 c;
#pragma unroll
    for (int i = 0; i < N; i++) c.v[i] = CMEM(i);
    return unpack(canonical(mul(a, c)));
}

// a^(p-2) (4-bit fixed windows, rolled loops); a of up to a few p, one lazy operand, a != 0 mod p.
GRAPE_HD Fp30 inverse(const Fp30& a) {
    Fp30 tbl[16];
    tbl[0] = one();
    tbl[1] = mul(a, one());
    for (int i = 2; i < 16; i++) tbl[i] = mul(tbl[i - 1], tbl[1]);
    Fp30 acc = one();
    bool started = false;
    for (int limb = FW - 1; limb >= 0; limb--) {
        uint32_t e = 0;
        for (int k = 0; k < FW; k++) e = (k == limb) ? FpParams::pm2(k) : e;
        for (int nib = 7; nib >= 0; nib--) {
            if (started) {
                acc = sqr(acc);
                acc = sqr(acc);
                acc = sqr(acc);
                acc = sqr(acc);
            }
            uint32_t w = (e >> (4 * nib)) & 15u;
            if (w) {
                acc = mul(acc, tbl[w]);
                started = true;
            }
        }
    }
    return acc;
}

// ------------------------------------------------------------------------------------------------
// Modular inversion by divsteps (divstep.hpp), whose limbs are of 30 bits too: about 800 divsteps for a 381-bit
// modulus, i.e. some 27 batches of a few hundred instructions each - one inversion sits on the
// critical path of every row epilogue.
// ------------------------------------------------------------------------------------------------
namespace by {

using divstep::M30;
using divstep::Mat;
using divstep::divsteps30;

constexpr int L = N;

#if defined(GRAPE_CURVE_BN254)
constexpr uint32_t PINV30 = 0x1b799c77u;    // p^-1 mod 2^30
GRAPE_HD int32_t P30(int i) {
    constexpr int32_t t[9] = {0x187cfd47, 0x3082305b, 0x071ca8d3, 0x205aa45a, 0x01585d97,
                              0x0116da06, 0x1a029b85, 0x139cb84c, 0x00003064};
    return t[i];
}
#else
constexpr uint32_t PINV30 = 0x00030003u;    // p^-1 mod 2^30
GRAPE_HD int32_t P30(int i) {
    constexpr int32_t t[13] = {0x3fffaaab, 0x27fbffff, 0x153ffffb, 0x2affffac, 0x30f6241e, 0x034a83da, 0x112bf673,
                               0x12e13ce1, 0x2cd76477, 0x1ed90d2e, 0x29a4b1ba, 0x3a8e5ff9, 0x001a0111};
    return t[i];
}
#endif
struct PMod {
    static constexpr uint32_t INV30 = PINV30;
    static GRAPE_HD int32_t limb(int i) { return P30(i); }
};
// 1110 divsteps at most for 384 bits, 741 for 256 bits
constexpr int kBatches = divstep::batches_for_bits(32 * FpParams::N);

GRAPE_HD void update_fg(int32_t* f, int32_t* g, const Mat& t) { divstep::update_fg<L>(f, g, t); }
GRAPE_HD void update_de(int32_t* d, int32_t* e, const Mat& t) { divstep::update_de<L, PMod>(d, e, t); }

}  // namespace by

// 1/a in Montgomery form (radix R') for a of up to a few p, one lazy operand, a != 0 mod p; a product.
GRAPE_HD Fp30 inverse_by(const Fp30& a) {
    using namespace by;
    // canonical integer of a (still carrying the Montgomery factor) in [0, p)
    const Fp30 t = canonical(mul(a, one()));
    int32_t f[L], g[L], d[L], e[L];
#pragma unroll
    for (int k = 0; k < L; k++) {
        g[k] = t.v[k];
        f[k] = P30(k);
        d[k] = 0;
        e[k] = 0;
    }
    e[0] = 1;
    int32_t delta = 1;
    for (int batch = 0; batch < kBatches; batch++) {
        uint32_t gz = 0;
#pragma unroll
        for (int k = 0; k < L; k++) gz |= (uint32_t)g[k];
        if (gz == 0) break;
        Mat m;
        delta = divsteps30(delta, (uint32_t)f[0] | ((uint32_t)f[1] << 30), (uint32_t)g[0] | ((uint32_t)g[1] << 30), m);
        update_de(d, e, m);
        update_fg(f, g, m);
    }
    // now g = 0, f = +-1 and d * a = f (mod p): the inverse is d * f, in (-2p, 2p), |limbs| <= 2^30
    const int32_t fneg = f[L - 1] >> 31;          // all-ones when f = -1
    Fp30 x, r3;
#pragma unroll
    for (int k = 0; k < L; k++) {
        x.v[k] = (d[k] ^ fneg) - fneg;            // limb-wise negation when f = -1
        r3.v[k] = R3(k);
    }
    return mul(x, r3);
}

}  // namespace fp30

// ------------------------------------------------------------------------------------------------
// XYZZ accumulator in the working form.  Invariants between additions: all coordinates balanced, zz below p, zz and zzz
// never congruent to zero, |x| < 3.5p, |y| and zzz below p; on BN254, where a product in wide digits reaches 1.4p,
// |x| < 5.7p (R^2 less PPP and 2Q) and zzz < 1.4p.  `inf` marks the identity.  All of the values below stay under 14 p (BN254: 23 p),
// all products of them far under 630 p^2 (86000 p^2).
// ------------------------------------------------------------------------------------------------
struct Xyzz30 {
    Fp30 x, y, zz, zzz;
    bool inf;
};
struct Affine30 {   // coordinates in (-p, p), balanced
    Fp30 x, y;
};

GRAPE_HD Xyzz30 xyzz30_inf() {
    Xyzz30 r;
    r.x = fp30::zero();
    r.y = fp30::zero();
    r.zz = fp30::zero();
    r.zzz = fp30::zero();
    r.inf = true;
    return r;
}

GRAPE_HD G1Xyzz xyzz30_to_canonical(const Xyzz30& a) {
    if (a.inf) return G1Xyzz::inf();
    G1Xyzz r;
    r.x = fp30::to_canonical(a.x);
    r.y = fp30::to_canonical(a.y);
    r.zz = fp30::to_canonical(a.zz);
    r.zzz = fp30::to_canonical(a.zzz);
    return r;
}
GRAPE_HD Xyzz30 xyzz30_from_canonical(const G1Xyzz& a) {
    Xyzz30 r;
    r.inf = a.is_inf();
    r.x = fp30::from_canonical(a.x);
    r.y = fp30::from_canonical(a.y);
    r.zz = fp30::from_canonical(a.zz);
    r.zzz = fp30::from_canonical(a.zzz);
    return r;
}

// acc += (negate ? -p : p) for a finite affine point p (the caller skips the identity).
// Returns false when the addition is one of the exceptional cases (p = +-acc): then acc is left
// untouched and the caller must take the exact slow path.
GRAPE_HD bool xyzz30_madd(Xyzz30& acc, const Affine30& p, bool negate) {
    using namespace fp30;
    const Fp30 py = cneg(p.y, negate);
    if (acc.inf) {
        acc.x = p.x;
        acc.y = py;
        acc.zz = one();
        acc.zzz = one();
        acc.inf = false;
        return true;
    }
    const Fp30 Pd = mulb_less(p.x, acc.zz, acc.x);      // U2 - X1
    const Fp30 R = mulb_less(py, acc.zzz, acc.y);       // S2 - Y1
    const Fp30 PP = sqr(Pd);
    const Fp30 ZZ3 = mulb_below_p(acc.zz, PP);
    if (is_zero(ZZ3)) return false;                    // PP = 0  <=>  P = 0: doubling or cancellation
    const Fp30 PPP = mulb(Pd, PP);
    const Fp30 Q = mulb(acc.x, PP);
    const Fp30 X3 = sqr_less(R, PPP, Q);
    const Fp30 T = balance(sub(Q, X3));
    const Fp30 Y3 = mul_sub(R, T, acc.y, PPP);
    acc.zzz = mulb(acc.zzz, PPP);
    acc.zz = ZZ3;
    acc.x = X3;
    acc.y = Y3;
    return true;
}

// acc <- 2 * acc (curve with a = 0, 6M + 3S: U = 2Y, V = U^2, W = U V, S = X V,
// M = 3 X^2, X3 = M^2 - 2S, Y3 = M (S - X3) - W Y, ZZ3 = V ZZ, ZZZ3 = W ZZZ).  No exceptional case on
// a group of odd prime order; the identity stays the identity.
GRAPE_HD void xyzz30_dbl(Xyzz30& acc) {
    using namespace fp30;
    if (acc.inf) return;
    Fp30 U;
#pragma unroll
    for (int i = 0; i < N; i++) U.v[i] = 2 * acc.y.v[i];
    U = balance(U);
    const Fp30 V = sqr(U);
    const Fp30 Wd = mulb(U, V);
    const Fp30 S = mulb(acc.x, V);
    const Fp30 X2 = sqr(acc.x);
    Fp30 M;
#pragma unroll
    for (int i = 0; i < N; i++) M.v[i] = 3 * X2.v[i];
    M = balance<true>(M);
    const Fp30 X3 = sqr_less(M, zero(), S);
    const Fp30 T = balance(sub(S, X3));
    const Fp30 Y3 = mul_sub(M, T, Wd, acc.y);
    acc.zz = mulb(V, acc.zz);
    acc.zzz = mulb(Wd, acc.zzz);
    acc.x = X3;
    acc.y = Y3;
}

// acc += q, both accumulators in the working form (12M + 2S).  Returns false, leaving acc
// untouched, in the exceptional cases q = +-acc; identities are handled here.
GRAPE_HD bool xyzz30_add(Xyzz30& acc, const Xyzz30& q) {
    using namespace fp30;
    if (q.inf) return true;
    if (acc.inf) {
        acc = q;
        return true;
    }
    const Fp30 U1 = mulb(acc.x, q.zz);
    const Fp30 S1 = mulb(acc.y, q.zzz);
    const Fp30 Pd = mulb_less(q.x, acc.zz, U1);         // U2 - U1
    const Fp30 R = mulb_less(q.y, acc.zzz, S1);         // S2 - S1
    const Fp30 PP = sqr(Pd);
    const Fp30 ZZ3 = mulb_below_p(mulb(acc.zz, q.zz), PP);
    if (is_zero(ZZ3)) return false;
    const Fp30 PPP = mulb(Pd, PP);
    const Fp30 Q = mulb(U1, PP);
    const Fp30 X3 = sqr_less(R, PPP, Q);
    const Fp30 T = balance(sub(Q, X3));
    const Fp30 Y3 = mul_sub(R, T, S1, PPP);
    acc.zzz = mulb(mulb(acc.zzz, q.zzz), PPP);
    acc.zz = ZZ3;
    acc.x = X3;
    acc.y = Y3;
    return true;
}

// affine image in canonical 32-bit form; the identity maps to (0,0)
GRAPE_HD G1Affine xyzz30_to_affine(const Xyzz30& a) {
    using namespace fp30;
    if (a.inf) return G1Affine::inf();
    const Fp30 zzz_inv = inverse_by(a.zzz);
    const Fp30 zinv = mul(zzz_inv, a.zz);             // 1/Z
    G1Affine r;
    r.x = to_canonical(mul(a.x, sqr(zinv)));
    r.y = to_canonical(mul(a.y, zzz_inv));
    return r;
}

// ------------------------------------------------------------------------------------------------
// Affine + affine with the inversion supplied by the caller (Montgomery's trick over many
// independent additions: table generation).  Inputs are finite points with balanced coordinates in (-p, p).
// ------------------------------------------------------------------------------------------------
// a normalised value in [0, 4p) -> the representative in [0, p)
GRAPE_HD Fp30 fp30_below_p(Fp30 t) {
#pragma unroll
    for (int s = 1; s >= 0; s--) {
        Fp30 d;
#pragma unroll
        for (int i = 0; i < fp30::N; i++) d.v[i] = t.v[i] - (s ? fp30::P2(i) : fp30::P(i));
        d = fp30::normalize(d);
        const bool ok = d.v[fp30::N - 1] >= 0;
#pragma unroll
        for (int i = 0; i < fp30::N; i++) t.v[i] = ok ? d.v[i] : t.v[i];
    }
    return t;
}
// denominator of the slope of e + f (x_e - x_f), or of 2 e (2 y_e) when `dbl`; a value congruent
// to zero means that the sum is no finite affine addition (e = +-f, or a point of order two)
GRAPE_HD Fp30 affine30_slope_den(const Affine30& e, const Affine30& f, bool dbl) {
    Fp30 r;
#pragma unroll
    for (int i = 0; i < fp30::N; i++) r.v[i] = dbl ? 2 * e.y.v[i] : e.x.v[i] - f.x.v[i];
    return r;
}
// e + f (2 e when `dbl`; then e must equal f) given dinv = 1 / affine30_slope_den(e, f, dbl), a
// product: 3M + 1S (one more S for the doubling), coordinates in [0, p), normalised
GRAPE_HD Affine30 affine30_add_given_inverse(const Affine30& e, const Affine30& f, bool dbl, const Fp30& dinv) {
    using namespace fp30;
    Fp30 num;
    if (dbl) {
        const Fp30 xx = sqr(e.x);       // (of f, which a run of additions keeps, the limb products are kept in registers too)
#pragma unroll
        for (int i = 0; i < N; i++) num.v[i] = 3 * xx.v[i];
        num = balance<true>(num);
    } else {
        num = sub(e.y, f.y);
    }
    const Fp30 lam = mul(num, dinv);
    const Fp30 ll = sqr_below_p(lam);
    Fp30 x3;
#pragma unroll
    for (int i = 0; i < N; i++) x3.v[i] = ll.v[i] - e.x.v[i] - f.x.v[i] + P3(i);   // in (0, 4p) for coordinates in [0, p)
    x3 = fp30_below_p(normalize(x3));
    const Fp30 ly = mul(lam, balance(sub(e.x, x3)));
    Fp30 y3;
#pragma unroll
    for (int i = 0; i < N; i++) y3.v[i] = ly.v[i] - e.y.v[i] + P2(i);              // in (0, 3p)
    Affine30 r;
    r.x = x3;
    r.y = fp30_below_p(normalize(y3));
    return r;
}

}  // namespace grape
