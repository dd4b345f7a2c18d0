// Group operations on four lanes: lane 4q + r of a wave holds coordinate r of an XYZZ accumulator of
// fp30.hpp (x, y, zz, zzz).
//
// Why: the last steps of a commitment - the row sums, the map to affine coordinates, the one row of an
// opening - are latency chains, and a lone wave issues an instruction about every 8 cycles here.  One
// lane's general addition is 5600 instructions long (14 products); its products fall into four groups
// of up to four independent ones, so a quad takes four products' time (about 2200 instructions), holds
// 14 registers of state instead of 53 and runs a fraction of the code.
// The price is throughput: 140 instead of 88 wave instructions per addition, so the accumulation
// kernels, which fill the chip, keep one lane per accumulator.
//
// Every lane of a quad must be active and take the same branch.
#pragma once
#include "fp30.hpp"

namespace grape {
namespace quad {

// lane r of a quad receives the value of lane (CTRL >> 2r) & 3
template <int CTRL>
__device__ __forceinline__ int32_t perm(int32_t x) {
    return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ Fp30 perm(const Fp30& a) {
    Fp30 r;
#pragma unroll
    for (int i = 0; i < fp30::N; i++) r.v[i] = perm<CTRL>(a.v[i]);
    return r;
}
constexpr int ctrl(int a, int b, int c, int d) { return a | (b << 2) | (c << 4) | (d << 6); }
constexpr int kFrom0 = ctrl(0, 0, 0, 0), kFrom1 = ctrl(1, 1, 1, 1), kCross = ctrl(2, 3, 0, 1), kPair = ctrl(1, 0, 3, 2);

// all-ones in the lanes of coordinate K.  Masks and v_bfi instead of conditions: from conditions the compiler makes
// branches around single limbs.
template <int K>
__device__ __forceinline__ int32_t lanes() {
    int32_t m = (threadIdx.x & 3) == K ? -1 : 0;
    asm("" : "+v"(m));
    return m;
}
__device__ __forceinline__ int32_t select(int32_t mask, int32_t a, int32_t b) { return (a & mask) | (b & ~mask); }
__device__ __forceinline__ Fp30 select(int32_t mask, const Fp30& a, const Fp30& b) {
    Fp30 r;
#pragma unroll
    for (int i = 0; i < fp30::N; i++) r.v[i] = select(mask, a.v[i], b.v[i]);
    return r;
}

struct Acc {          // one lane's coordinate of a quad's accumulator
    Fp30 v;           // balanced; values per coordinate as for Xyzz30 (|y| below 2p)
    bool inf;         // the same in all four lanes
};
__device__ __forceinline__ Acc identity() {
    Acc a;
    a.v = fp30::zero();
    a.inf = true;
    return a;
}

// acc <- 2 acc (the formulas of xyzz30_dbl): three products' time
__device__ __forceinline__ void dbl(Acc& acc) {
    using namespace fp30;
    if (acc.inf) return;
    const int32_t m0 = lanes<0>(), m1 = lanes<1>(), m2 = lanes<2>(), m3 = lanes<3>();
    // lane 0: X^2, lane 1: V = (2Y)^2
    Fp30 w;
#pragma unroll
    for (int i = 0; i < N; i++) w.v[i] = acc.v.v[i] + (acc.v.v[i] & m1);
    w = balance(w);
    const Fp30 s1 = sqr(w);                                   // lanes 2, 3 unused
    const Fp30 V = perm<kFrom1>(s1);
    Fp30 M = perm<kFrom0>(s1);
#pragma unroll
    for (int i = 0; i < N; i++) M.v[i] = 3 * M.v[i];
    M = balance<true>(M);
    // lane 0: S = X V, lane 1: W = 2Y V, lane 2: ZZ V, lane 3: M^2
    const Fp30 s2 = mulb(select(m3, M, w), select(m3, M, V));
    const Fp30 MM = perm<ctrl(3, 3, 3, 3)>(s2);
    const Fp30 Wd = perm<kFrom1>(s2);
    Fp30 X3;                                                  // only lane 0's is used
#pragma unroll
    for (int i = 0; i < N; i++) X3.v[i] = MM.v[i] - 2 * s2.v[i];
    X3 = balance<true>(X3);
    // lane 0: M (S - X3), lane 1: W Y, lane 3: W ZZZ
    const Fp30 s3 = mul(select(m0, M, Wd), select(m0, sub(s2, X3), acc.v));      // one lazy operand
    const Fp30 y0 = perm<kFrom0>(s3);
    Fp30 y3;
#pragma unroll
    for (int i = 0; i < N; i++) y3.v[i] = y0.v[i] - s3.v[i];
    y3 = balance(y3);
    acc.v = select(m0, X3, select(m1, y3, select(m2, s2, s3)));
}

// acc += q (the formulas of xyzz30_add, every exceptional case included): four products' time
__device__ __forceinline__ void add(Acc& acc, const Acc& q) {
    using namespace fp30;
    if (q.inf) return;
    if (acc.inf) {
        acc = q;
        return;
    }
    const int32_t m0 = lanes<0>(), m1 = lanes<1>(), m2 = lanes<2>(), m01 = m0 | m1;
    // U1 = X1 ZZ2, S1 = Y1 ZZZ2, U2 = ZZ1 X2, S2 = ZZZ1 Y2
    const Fp30 t = mulb(acc.v, perm<kCross>(q.v));
    const Fp30 D = balance(sub(perm<kCross>(t), t));          // lanes 0, 1: P = U2 - U1, R = S2 - S1
    // P^2, R^2, ZZ1 ZZ2, ZZZ1 ZZZ2
    const Fp30 s2 = mulb_below_p(select(m01, D, acc.v), select(m01, D, q.v));
    const int zero = is_zero(s2) ? 1 : 0;
    if (perm<kFrom0>(zero)) {                                 // q = +-acc
        if (perm<kFrom1>(zero)) dbl(acc);
        else acc = identity();
        return;
    }
    const Fp30 PP = perm<kFrom0>(s2);
    // PPP, Q = U1 PP, ZZ3
    const Fp30 s3 = mulb(select(m0, D, select(m1, perm<kFrom0>(t), s2)), PP);
    const Fp30 PPP = perm<kFrom0>(s3);
    Fp30 X3;                                                  // only lane 1's is used: R^2 - PPP - 2Q
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < N; i++) {                             // balanced as in balance(); a limb may pass 2^31, its half does not
        const int32_t x = s2.v[i] - PPP.v[i];
        const uint32_t limb = (uint32_t)x - 2 * (uint32_t)s3.v[i];
        X3.v[i] = (i < N - 1 ? low30(limb) : (int32_t)limb) + c;
        c = ((x >> 1) - s3.v[i] + HALF / 2) >> (W - 1);
    }
    // S1 PPP, R (Q - X3), -, ZZZ1 ZZZ2 PPP
    const Fp30 T = sub(s3, X3);                               // lazy
    const Fp30 s4 = mul(select(m0, perm<kFrom1>(t), select(m1, D, s2)), select(m1, T, PPP));
    const Fp30 sp = perm<kFrom0>(s4), x3 = perm<kFrom1>(X3);
    Fp30 y3;
#pragma unroll
    for (int i = 0; i < N; i++) y3.v[i] = s4.v[i] - (sp.v[i] & m1);
    acc.v = select(m0, x3, select(m2, s3, balance(y3)));
}

// 30 divsteps on the low words f, g (lane 0: x1 = f, x2 = g), the columns of the transition matrix in the same registers
// of the other lanes (lane 1: x1 = u, x2 = q from 1, 0; lane 2: x1 = v, x2 = r from 0, 1).  divsteps30 of divstep.hpp with
// one kind of operation for all of them: g is not halved, f is doubled instead like u and v, and step i
// looks at bit i of g.  12 instructions a step where one lane takes 26.
__device__ __forceinline__ int32_t divsteps30(int32_t delta, int32_t& x1, int32_t& x2) {
    int32_t nd = -delta;
#pragma unroll
    for (int i = 0; i < 30; i++) {
        const int32_t g = perm<kFrom0>(x2);
        const int32_t odd = (int32_t)((uint32_t)g << (31 - i)) >> 31;             // all-ones when g is odd
        const int32_t swap = odd & (nd >> 31);
        const int32_t n1 = select(swap, x2, x1), n2 = select(swap, -x1, x2);      // (f, g) <- (g, -f)
        x2 = n2 + (n1 & odd);                                                     // -f is odd too: g is made even
        x1 = (int32_t)((uint32_t)n1 << 1);
        nd = (nd ^ swap) + ~swap;                                                 // delta <- 1 -+ delta
    }
    return -nd;
}

// 1/a for the same a in all four lanes (up to a few p, not 0 mod p); a product, the same in all
// four lanes.  inverse_by of fp30.hpp with one of the vectors f, g, d, e per lane: a batch's update of the
// four vectors is one row of multiply-adds instead of four.
__device__ __forceinline__ Fp30 inverse_by(const Fp30& a) {
    using namespace fp30;
    using namespace fp30::by;
    const int32_t m0 = lanes<0>(), m1 = lanes<1>(), m2 = lanes<2>(), m3 = lanes<3>();
    const Fp30 t = canonical(fp30::mul(a, one()));            // integer in [0, p), still with the Montgomery factor
    int32_t x[L];                                             // lane 0: f, 1: g, 2: d, 3: e
#pragma unroll
    for (int k = 0; k < L; k++) x[k] = (P30(k) & m0) | (t.v[k] & m1) | (k == 0 ? m3 & 1 : 0);
    int32_t delta = 1;
    const int32_t de = m2 | m3, ge = m1 | m3;
    for (int batch = 0; batch < kBatches; batch++) {
        uint32_t z = 0;
#pragma unroll
        for (int k = 0; k < L; k++) z |= (uint32_t)x[k];
        if (perm<kFrom1>((int32_t)z) == 0) break;             // g = 0
        const uint32_t lo = (uint32_t)x[0] | ((uint32_t)x[1] << 30);
        int32_t x1 = (perm<kFrom0>((int32_t)lo) & m0) | (m1 & 1), x2 = (perm<kFrom1>((int32_t)lo) & m0) | (m2 & 1);
        delta = quad::divsteps30(delta, x1, x2);
        // f' = u f + v g, g' = q f + r g (d', e' alike, plus the multiple of p that clears the low 30 bits)
        const int32_t u = perm<kFrom1>(x1), q = perm<kFrom1>(x2), v = perm<ctrl(2, 2, 2, 2)>(x1), w = perm<ctrl(2, 2, 2, 2)>(x2);
        const int32_t own = select(ge, w, u), other = select(ge, q, v);
        const int32_t sx = x[L - 1] >> 31, sy = perm<kPair>(sx);
        int32_t md = (own & sx) + (other & sy);
        int64_t c = (int64_t)own * x[0] + (int64_t)other * perm<kPair>(x[0]);
        md -= (int32_t)((PINV30 * (uint32_t)c + (uint32_t)md) & (uint32_t)M30);
        md &= de;
        c += (int64_t)P30(0) * md;
        c >>= 30;
#pragma unroll
        for (int i = 1; i < L; i++) {
            c += (int64_t)own * x[i] + (int64_t)other * perm<kPair>(x[i]) + (int64_t)P30(i) * md;
            x[i - 1] = (int32_t)c & M30;
            c >>= 30;
        }
        x[L - 1] = (int32_t)c;
    }
    // g = 0, f = +-1, d * a = f (mod p): d, in (-2p, p) with limbs below 2^30, to every lane, negated when f = -1
    const int32_t fneg = perm<kFrom0>(x[L - 1]) >> 31;
    Fp30 out, r3;
#pragma unroll
    for (int k = 0; k < L; k++) {
        const int32_t d = perm<ctrl(2, 2, 2, 2)>(x[k]);
        out.v[k] = (d ^ fneg) - fneg;
        r3.v[k] = R3(k);
    }
    return fp30::mul(out, r3);
}

__device__ __forceinline__ void cneg(Acc& a, bool flag) {
    const int32_t m = lanes<1>() & (flag ? -1 : 0);
#pragma unroll
    for (int i = 0; i < fp30::N; i++) a.v.v[i] = (a.v.v[i] ^ m) - m;
}

// affine image in canonical 32-bit form: lane 0 returns x, lane 1 returns y (zero for the identity); lanes 2, 3 nothing of use
__device__ __forceinline__ Fp to_affine(const Acc& a) {
    using namespace fp30;
    if (a.inf) return Fp::zero();
    const Fp30 zzz_inv = quad::inverse_by(perm<ctrl(3, 3, 3, 3)>(a.v));
    const Fp30 zinv = mul(zzz_inv, perm<ctrl(2, 2, 2, 2)>(a.v));      // 1/Z
    return to_canonical(mul(a.v, select(lanes<0>(), sqr(zinv), zzz_inv)));
}

}  // namespace quad
}  // namespace grape
