// Long weighted rounds that carry their weights in one of the tensors.
//
// A round over index pairs g sums e_g (a0 + t da)(s0 + t ds) with e_g = eq(u, g); weighing costs two reduced products a pair, as
// much as everything else (wround2_kernel).  But the next round's weights are this one's without the factor of one
// variable: e_(b, g') = e_g' f_b with f_0 = 1 - u_j, f_1 = u_j for the top bit b.  So the first round stores the weighted fold
// Z_g = e_g S'_g in the place of S', and from then on
//   q(0) = sum a0 Z0 / f_0,   q(1) = sum a1 Z1 / f_1,   Z' = Z0 + k Z1   with k = v f_0 / (f_1 (1 - v)),
// up to a factor that the host keeps.  Two plain products and two folds a pair.  The third value that a round's polynomial
// of degree 2 needs is its value at the challenge, and that is the next round's q(0) f_0 + q(1) f_1: the host solves for it from
// the last round up.  Only the high variables' weights are carried (eq_high); those of the low ones, eq[l] with l the index
// modulo `period`, multiply a thread's sums once at the end as in wround2_kernel, and what is left in Z after the last
// long round is a factor per period.  Challenges and coordinates of the point that are 0 or 1 have no inverse: such proofs
// take wround2_kernel (the host asks).
//
// A lookup's first round has A (S + beta) = 1 at every index, so q(0) = q(1) = 1 and it sums nothing weighted (a table with an
// entry that has no inverse is refused by the table side's rounds, which sum B (T + beta)).  Gathered by
// index, its folds are sums of two table entries: v x1 + (1 - v) x0 with both multiples of every entry made before.
// Bound: instruction issue and HBM about evenly (a pair of later rounds is six elements, 192 bytes, at 4.7 TB/s).  Against
// wround2_kernel: the gathered first round of 2^26 pairs 2.8 -> 2.1 ms, a round of 2^25 pairs 1.77 -> 1.34 ms, the first
// round of a 2048 x 11008 element product 0.69 -> 0.61 ms and its second 0.36 -> 0.23 ms.  A thread's next operands are asked
// for before this pair's arithmetic: two waves a SIMD do not cover the loads (2048 x 11008 proof 1.33 -> 1.29 ms).
// Proofs run the rounds two to a pass (carried_pair_kernel), an odd one's last alone; a single first round, gathered or with the weights
// entering, is there for callers of grape_carried_queue.
#include "fr_device.hpp"

namespace grape {

constexpr int kCarriedIters = 24;

// halves[2 t], halves[2 t + 1] = (1 - v) B_t, (1 - v)(T_t + beta); halves[2 len + 2 t], [2 len + 2 t + 1] = v B_t, v (T_t + beta)
__global__ void __launch_bounds__(kBlock) carried_halves_kernel(uint32_t* halves, const uint32_t* B, const uint32_t* T, const uint32_t* beta,
                                                                const uint32_t* v, uint32_t len) {
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= len) return;
    const Fr vv = ld_fr(v, 0), b = ld_fr(B, t), s = add(ld_fr(T, t), ld_fr(beta, 0));
    const Fr vb = fr26::mulc(b, vv), vs = fr26::mulc(s, vv);
    st_fr(halves, 2 * (size_t)t, sub(b, vb));
    st_fr(halves, 2 * (size_t)t + 1, sub(s, vs));
    st_fr(halves, 2 * ((size_t)len + t), vb);
    st_fr(halves, 2 * ((size_t)len + t) + 1, vs);
}

struct CarriedSpan {
    size_t first, stride;
    uint32_t h, low, hstep;
};
// a thread keeps one index modulo the period and steps over whole periods
__device__ __forceinline__ CarriedSpan carried_span(uint32_t period, uint32_t hstep) {
    CarriedSpan s;
    s.first = (size_t)blockIdx.x * kBlock + threadIdx.x;
    s.hstep = hstep;
    s.stride = (size_t)hstep * period;
    s.h = (uint32_t)s.first / period;
    s.low = (uint32_t)s.first - s.h * period;
    return s;
}

// First round of a lookup, gathered: A_out = the folded A, Z_out = eq_high[h] (S + beta folded); partial: the two halves' plain
// sums, times 1 - v and v.
// 2^26 pairs take 2.1 ms at three, four or five waves a SIMD, 2.6 at six (spills); indices asked for one step ahead: 2.4.
__global__ void __launch_bounds__(kBlock, 2) carried_gather_kernel(uint32_t* A_out, uint32_t* Z_out, const int32_t* __restrict__ idx1,
                                                                   const uint32_t* halves, uint32_t len, const uint32_t* Eh, uint32_t period,
                                                                   uint32_t hstep, uint32_t n_out, uint32_t* partial) {
    __shared__ Fr lds[2 * (kBlock / 64)];
    const CarriedSpan sp = carried_span(period, hstep);
    fr26::Limbs sb0, sb1;                       // 24 terms below 2^26
#pragma unroll
    for (int k = 0; k < fr26::N; k++) sb0.v[k] = sb1.v[k] = 0;
    uint32_t h = sp.h;
    for (size_t g = sp.first < sp.stride ? sp.first : n_out; g < n_out; g += sp.stride, h += sp.hstep) {
        const uint32_t j0 = (uint32_t)idx1[g], j1 = (uint32_t)idx1[g + n_out];         // 0 marks an element outside the table
        const size_t r0 = 2 * (size_t)(j0 ? j0 - 1 : 0), r1 = 2 * ((size_t)len + (j1 ? j1 - 1 : 0));
        const Fr b0 = ld_fr(halves, r0), s0 = ld_fr(halves, r0 + 1);
        const Fr b1 = ld_fr(halves, r1), s1 = ld_fr(halves, r1 + 1);
        const fr26::Limbs e16 = fr26::pack16(ld_fr(Eh, h));
        st_fr(A_out, g, add(b0, b1));
        sb0 = fr26::add(sb0, fr26::pack(b0));
        sb1 = fr26::add(sb1, fr26::pack(b1));
        st_fr(Z_out, g, fr26::unpack(fr26::canon(fr26::product(e16, fr26::pack(add(s0, s1)), 0), 1)));
    }
    Fr acc[2] = {fr26::limb_sum_to_fr(sb0, 0), fr26::limb_sum_to_fr(sb1, 0)};
    block_sum<2>(acc, lds);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < 2; k++) st_fr(partial, (size_t)blockIdx.x * 2 + k, acc[k]);
    }
}

// ENTER: the first round of an element product, Z is S itself and takes the weights on here (A and S of any reader: not
// written).  PLAIN: the plain sums of A's halves too.
template <bool ENTER, bool PLAIN>
__global__ void __launch_bounds__(kBlock, 2) carried_round_kernel(uint32_t* A_out, uint32_t* Z_out, const uint32_t* A, const uint32_t* Z,
                                                                  const uint32_t* E, const uint32_t* Eh, uint32_t period, uint32_t hstep,
                                                                  uint32_t n_out, const int32_t* __restrict__ tab_a, const int32_t* __restrict__ tab_z,
                                                                  uint32_t* partial) {
    constexpr int NV = PLAIN ? 4 : 2;
    __shared__ Fr lds[NV * (kBlock / 64)];
    const CarriedSpan sp = carried_span(period, hstep);
    fr26::Acc P0, P1;
    fr26::acc_zero(P0);
    fr26::acc_zero(P1);
    fr26::Limbs sa0, sa1;
#pragma unroll
    for (int k = 0; k < fr26::N; k++) sa0.v[k] = sa1.v[k] = 0;
    uint32_t h = sp.h;
    size_t g = sp.first < sp.stride ? sp.first : n_out;
    // the next index's operands are on their way while this one's are worked on (the last index asks for its own again)
    Fr na0, na1, nz0, nz1, ne;
    if (g < n_out) {
        na0 = ld_fr(A, g);
        na1 = ld_fr(A, g + n_out);
        nz0 = ld_fr(Z, g);
        nz1 = ld_fr(Z, g + n_out);
        if (ENTER) ne = ld_fr(Eh, h);
    }
    for (; g < n_out; g += sp.stride, h += sp.hstep) {
        const fr26::Limbs a0 = fr26::pack(na0), a1 = fr26::pack(na1);
        fr26::Limbs z0 = fr26::pack(nz0), z1 = fr26::pack(nz1);
        const size_t gn = g + sp.stride < n_out ? g + sp.stride : g;
        na0 = ld_fr(A, gn);
        na1 = ld_fr(A, gn + n_out);
        nz0 = ld_fr(Z, gn);
        nz1 = ld_fr(Z, gn + n_out);
        const fr26::Limbs e16 = ENTER ? fr26::pack16(ne) : fr26::Limbs{};
        if (ENTER) ne = ld_fr(Eh, gn == g ? h : h + hstep);
        st_fr(A_out, g, foldt1(tab_a, a0, fr26::sub(a1, a0)));
        if (PLAIN) {
            sa0 = fr26::add(sa0, a0);
            sa1 = fr26::add(sa1, a1);
        }
        if (ENTER) {
            z0 = fr26::product(e16, z0, 0);                 // (0, 1.46 r): the fold of two such stays below 3.5 r
            z1 = fr26::product(e16, z1, 0);
            st_fr(Z_out, g, foldt1(tab_a, z0, fr26::sub(z1, z0)));
        } else {
            st_fr(Z_out, g, foldt1(tab_z, z0, z1));
        }
        fr26::mac(P0, a0, z0);                              // below 1.46 r^2 each: 24 of them below 35.1 r^2, within r after the reduction
        fr26::mac(P1, a1, z1);
    }
    Fr acc[NV];
    const Fr el = ld_fr(E, sp.low);
    acc[0] = fr26::mulc(fr26::unpack(fr26::canon_wide(fr26::reduce(P0, 0))), el);
    acc[1] = fr26::mulc(fr26::unpack(fr26::canon_wide(fr26::reduce(P1, 0))), el);
    if (PLAIN) {
        acc[2] = fr26::limb_sum_to_fr(sa0, 0);
        acc[3] = fr26::limb_sum_to_fr(sa1, 0);
    }
    block_sum<NV>(acc, lds);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < NV; k++) st_fr(partial, (size_t)blockIdx.x * NV + k, acc[k]);
    }
}

// Two consecutive rounds in one pass: the challenges are known, so what the first round folds is worked on at once and a
// quarter of the elements is written instead of a half that the next pass reads again (per eight elements read, two written: 320
// bytes where two passes move 576).
// Elements x_(b, c, g), b the variable of the first round, c that of the second: the two halves of a wave share 32 indices g, lanes
// of half c hold x_(0, c, g) and x_(1, c, g) of both tensors.  Each lane makes the first round's two products and folds of its pair
// and one of the second round's two products - three accumulators in registers where a lane that did both rounds alone would need
// four and spill; then the halves swap (v_permlane32_swap) and the lower one folds A, the upper one Z, each through its own
// table in LDS.  What is folded again stays in limbs, not reduced (foldt1_limbs).
// Bound: instruction issue (1240 instructions a lane and index, 1700 where the weights enter) and the loads of the next index, which
// are asked for where registers allow, a fifth of an index ahead; HBM carries 2.6 to 3.5 TB/s.  Against two passes: 2^27 elements
// gathered 2.0 + 1.5 -> 1.87 ms (three waves a SIMD; two: 2.23) and the eight rounds behind them 1.5 -> 1.19, the first two rounds of a
// 2048 x 11008 element product 0.535 + 0.27 -> 0.625 and the six behind them 0.27 -> 0.225.
// kGather: a lookup's first round with the next one.  kEnter: an element product's, the weights enter.  kLater: neither.
enum { kLater, kEnter, kGather };
struct CarriedPair {
    uint32_t *A_out, *Z_out;
    const uint32_t *A, *Z;
    const int32_t* idx1;
    const uint32_t* halves;
    uint32_t len;
    const uint32_t *E, *Eh;
    uint32_t period, hstep, n_out;         // n_out: elements left after both rounds
    const int32_t *tab_a, *tab_z;          // first round
    const int32_t *next_a, *next_z;        // second round
    uint32_t *partial, *next_partial;
};
template <int MODE, bool PLAIN>
__global__ void __launch_bounds__(kBlock, MODE == kGather ? 3 : 2) carried_pair_kernel(CarriedPair p) {
    constexpr bool SUMS = MODE != kGather;                  // the first round has weighted sums
    constexpr int V0 = SUMS ? 2 : 0, NV = V0 + 1 + (PLAIN ? 2 : 0), NW = kBlock / 64;
    __shared__ Fr lds[NV * 2 * NW];
    constexpr int kTab = fr26::N * kFoldLdsRow, kTabs = MODE == kLater && PLAIN ? 3 : 2;    // the third one folds the plain sums
    __shared__ __attribute__((aligned(16))) int32_t tabs[kTabs * kTab];
    for (int i = threadIdx.x; i < kTabs * fr26::kFoldTableWords; i += kBlock) {
        const int t = i / fr26::kFoldTableWords, w = i % fr26::kFoldTableWords;
        tabs[t * kTab + w / fr26::N * kFoldLdsRow + w % fr26::N] = (t == 0 ? p.next_a : t == 1 ? p.next_z : p.tab_a)[w];
    }
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = lane >> 5;
    const uint32_t first = (blockIdx.x * NW + wave) * 32 + (lane & 31);
    const uint32_t stride = p.hstep * p.period, n = p.n_out;
    const uint32_t c0 = half * n;                           // this lane's two elements of index g: g + c0 and 2 n behind it
    uint32_t h = first / p.period + half * (n / p.period);
    const int32_t* tab2 = tabs + half * kTab;
    const int32_t diff = half ? 0 : -1;                     // A is folded by lo + v (hi - lo), Z by lo + k hi
    fr26::Acc P0, P1, Q;
    if (SUMS) {
        fr26::acc_zero(P0);
        fr26::acc_zero(P1);
    }
    fr26::acc_zero(Q);
    fr26::Limbs sa0, sa1;
#pragma unroll
    for (int k = 0; k < fr26::N; k++) sa0.v[k] = sa1.v[k] = 0;
    uint32_t g = first < stride ? first : n;
    Fr na0, na1, nz0, nz1;
    if (SUMS && g < n) {
        na0 = ld_fr(p.A, g + c0);
        na1 = ld_fr(p.A, (size_t)g + c0 + 2 * n);
        nz0 = ld_fr(p.Z, g + c0);
        nz1 = ld_fr(p.Z, (size_t)g + c0 + 2 * n);
    }
    for (; g < n; g += stride, h += p.hstep) {
        fr26::Limbs a, z;                                   // this half's elements of the second round
        if (MODE == kGather) {
            const uint32_t j0 = (uint32_t)p.idx1[g + c0], j1 = (uint32_t)p.idx1[(size_t)g + c0 + 2 * n];       // 0 marks an element outside the table
            const size_t r0 = 2 * (size_t)(j0 ? j0 - 1 : 0), r1 = 2 * ((size_t)p.len + (j1 ? j1 - 1 : 0));
            const Fr b0 = ld_fr(p.halves, r0), s0 = ld_fr(p.halves, r0 + 1);
            const Fr b1 = ld_fr(p.halves, r1), s1 = ld_fr(p.halves, r1 + 1);
            const fr26::Limbs e16 = fr26::pack16(ld_fr(p.Eh, h));
            const fr26::Limbs l0 = fr26::pack(b0), l1 = fr26::pack(b1);
            sa0 = fr26::add(sa0, l0);
            sa1 = fr26::add(sa1, l1);
            a = fr26::normalize(fr26::add(l0, l1));         // below 2 r
            z = fr26::product(e16, fr26::pack(add(s0, s1)), 0);     // (0, 1.46 r)
        } else {
            arrived(na0);
            arrived(na1);
            arrived(nz0);
            arrived(nz1);
            const fr26::Limbs a0 = fr26::pack(na0), a1 = fr26::pack(na1);
            fr26::Limbs z0 = fr26::pack(nz0), z1 = fr26::pack(nz1);
            if (PLAIN) {
                sa0 = fr26::add(sa0, a0);
                sa1 = fr26::add(sa1, a1);
            }
            if (MODE == kEnter) {
                const fr26::Limbs e16 = fr26::pack16(ld_fr(p.Eh, h));
                z0 = fr26::product(e16, z0, 0);             // (0, 1.46 r)
                z1 = fr26::product(e16, z1, 0);
            }
            a = foldt1_limbs(p.tab_a, a0, fr26::sub(a1, a0));
            fr26::mac(P0, a0, z0);                          // below 1.46 r^2 each: 24 of them below 35.1 r^2
            fr26::mac(P1, a1, z1);
            z = MODE == kEnter ? foldt1_limbs(p.tab_a, z0, fr26::sub(z1, z0)) : foldt1_limbs(p.tab_z, z0, z1);
            // the next index's operands, asked for where their registers are free: the second round's share covers the loads
            // (the last index asks for its own again)
            const uint32_t gn = g + stride < n ? g + stride : g;
            asm volatile("" : "+v"(z.v[0]));
            na0 = ld_fr(p.A, gn + c0);
            na1 = ld_fr(p.A, (size_t)gn + c0 + 2 * n);
            nz0 = ld_fr(p.Z, gn + c0);
            nz1 = ld_fr(p.Z, (size_t)gn + c0 + 2 * n);
        }
        fr26::mac(Q, a, z);                                 // a within (-0.5, 2) r, z within (-0.5, 1.96) r: 24 of them within (-24, 95) r^2
        // lower lanes (A, index 0) (Z, index 0), upper ones the same of index 1 -> lower A of both, upper Z of both
        fr26::Limbs lo, d;
#pragma unroll
        for (int k = 0; k < fr26::N; k++) {
            const auto s = __builtin_amdgcn_permlane32_swap((uint32_t)a.v[k], (uint32_t)z.v[k], false, false);
            lo.v[k] = (int32_t)s[0];
            d.v[k] = (int32_t)s[1] - (lo.v[k] & diff);
        }
        st_fr(half ? p.Z_out : p.A_out, g, foldt_lds(tab2, lo, d));
    }
    Fr acc[NV];
    const Fr el = ld_fr(p.E, first % p.period);
    if (SUMS) {
        acc[0] = fr26::mulc(fr26::unpack(fr26::canon_wide(fr26::reduce(P0, 0))), el);
        acc[1] = fr26::mulc(fr26::unpack(fr26::canon_wide(fr26::reduce(P1, 0))), el);
    }
    acc[V0] = fr26::mulc(fr26::unpack(fr26::canon_wide(fr26::reduce(Q, 1))), el);       // (0.3 r, 5 r)
    if (PLAIN) {
        acc[V0 + 1] = fr26::limb_sum_to_fr(sa0, 0);
        acc[V0 + 2] = fr26::limb_sum_to_fr(sa1, 0);
    }
    // sums of each half: lds[value][half][wave]
#pragma unroll
    for (int k = 0; k < NV; k++) {
#pragma unroll
        for (int off = 16; off >= 1; off >>= 1) acc[k] = add(acc[k], shfl_down_fr(acc[k], off));
        if ((lane & 31) == 0) lds[(k * 2 + half) * NW + wave] = acc[k];
    }
    __syncthreads();
    const uint32_t t = threadIdx.x;
    Fr sum = Fr::zero();
    if (t < 2 * NV) {
        sum = lds[t * NW];
        for (int w = 1; w < NW; w++) sum = add(sum, lds[t * NW + w]);
    }
    __syncthreads();
    if (t < 2 * NV) lds[t] = sum;                           // [value][half]
    __syncthreads();
    // the first round's sums are over both halves; the second one's are the halves' own: of the products, and of A folded
    constexpr int NV0 = V0 + (PLAIN ? 2 : 0), NV1 = 2 + (PLAIN ? 2 : 0);
    if (t < NV0) {
        const int k = (int)t < V0 ? t : t + 1;
        st_fr(p.partial, (size_t)blockIdx.x * NV0 + t, add(lds[2 * k], lds[2 * k + 1]));
    } else if (t >= 64 && t < 64 + NV1) {
        const int k = t - 64, c = k & 1;
        Fr r = lds[2 * V0 + c];
        if (PLAIN && k >= 2) {
            const Fr s0 = lds[2 * (V0 + 1) + c], s1 = lds[2 * (V0 + 2) + c];
            if (MODE == kGather) r = add(s0, s1);
            else {
                const fr26::Limbs l = fr26::pack(s0);
                r = foldt_lds(tabs + 2 * kTab, l, fr26::sub(fr26::pack(s1), l));
            }
        }
        st_fr(p.next_partial, (size_t)blockIdx.x * NV1 + k, r);
    }
}

constexpr uint32_t kMaxCarried = 32;
struct CarriedFinish {
    const uint32_t* partial[kMaxCarried];
    uint32_t nblocks[kMaxCarried];
    uint32_t* out[kMaxCarried];
};
// NW weighted sums go to out[0 ..), times the radix factor 16 that they leave their kernel without, NV - NW plain ones to out[3 ..)
template <int NV, int NW, int BLOCK>
__global__ void __launch_bounds__(BLOCK) carried_final_kernel(CarriedFinish f) {
    __shared__ uint32_t lds9[NV * (BLOCK / 64) * 9];
    Fr tot[NV];
    workgroup_totals<NV, BLOCK>(tot, f.partial[blockIdx.x], f.nblocks[blockIdx.x], lds9);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < NV; k++) {
            Fr t = tot[k];
            if (k < NW) {
#pragma unroll
                for (int d = 0; d < 4; d++) t = add(t, t);
            }
            st_fr(f.out[blockIdx.x], k < NW ? k : 3 + k - NW, t);
        }
    }
}

// out[i] = Z[i] * factor[i / period] - beta
__global__ void __launch_bounds__(kBlock) carried_end_kernel(uint32_t* out, const uint32_t* Z, uint32_t n, const uint32_t* factor, uint32_t period,
                                                             const uint32_t* beta) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const Fr s = fr26::mulc(ld_fr(Z, i), ld_fr(factor, i / period));
    st_fr(out, i, beta ? sub(s, ld_fr(beta, 0)) : s);
}

// Periods a launch's threads step over: about four workgroups on a CU (an even number of waves on every SIMD and no last wave that
// is nearly empty), at most kCarriedIters indices a thread.
static uint32_t carried_hstep(uint32_t n_out, uint32_t period) {
    const uint32_t periods = n_out / period;
    uint32_t hstep = (uint32_t)(kNumCU * 4 * kBlock) / period;
    if (hstep < 1) hstep = 1;
    while ((periods + hstep - 1) / hstep > kCarriedIters) hstep *= 2;
    return hstep < periods ? hstep : periods;
}
// The same for a pass over two rounds, which has two threads for an index: as many rounds of two workgroups a CU as take
// the fewest steps, with kCarriedEnds of them for a workgroup's table, reductions and sums (the first pass
// of a 2048 x 11008 element product: 23 rows a step and 23 steps in 3.9 rounds, not 22 and 24 in 3.7).
constexpr uint32_t kCarriedEnds = 3;
static uint32_t carried_pair_hstep(uint32_t n_out, uint32_t period) {
    const uint32_t periods = n_out / period, slots = kNumCU * 2 * (kBlock / 2);      // indices in flight
    uint32_t best = periods, least = ~0u;
    for (uint32_t rounds = 1;; rounds++) {
        const uint64_t fit = (uint64_t)slots * rounds / period;
        const uint32_t hstep = fit < 1 ? 1 : fit < periods ? (uint32_t)fit : periods;
        const uint32_t steps = (periods + hstep - 1) / hstep;
        const uint32_t cost = ((uint32_t)(((uint64_t)hstep * period + slots - 1) / slots)) * (steps + kCarriedEnds);
        if (steps <= kCarriedIters && cost < least) {
            least = cost;
            best = hstep;
        }
        if (hstep == periods || steps <= kCarriedEnds) return best;
    }
}
// elements left after the pass that a round is part of
static uint32_t carried_pass_out(const grape_carried_args& a) { return a.pair == GRAPE_CARRIED_FIRST ? a.n_out / 2 : a.n_out; }
static uint32_t carried_step(const grape_carried_args& a) {
    if (a.pair == GRAPE_CARRIED_SINGLE) return carried_hstep(a.n_out, a.period);
    return carried_pair_hstep(carried_pass_out(a), a.period);
}
static unsigned carried_blocks(const grape_carried_args& a) {
    const size_t indices = (size_t)carried_step(a) * a.period;
    return blocks_for(a.pair == GRAPE_CARRIED_SINGLE ? indices : 2 * ((indices + 31) / 32 * 32));
}
static int carried_values(const grape_carried_args& a) { return a.idx1 ? 2 : a.plain_sums ? 4 : 2; }

}  // namespace grape

using namespace grape;

extern "C" {

int grape_carried_halves(uint32_t* halves, const uint32_t* B, const uint32_t* T, const uint32_t* beta, const uint32_t* v, uint32_t len, grape_stream_t st) {
    CHECK_PTR16(halves); CHECK_PTR16(B); CHECK_PTR16(T); CHECK_PTR16(beta); CHECK_PTR16(v);
    GRAPE_REQUIRE(len >= 1, "empty table");
    carried_halves_kernel<<<blocks_for(len), kBlock, 0, as_stream(st)>>>(halves, B, T, beta, v, len);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

static bool carried_shape_ok(const grape_carried_args* a) {
    if (!a || a->period < 1 || a->period > GRAPE_WROUND_MAX_PERIOD || a->pair > GRAPE_CARRIED_SECOND) return false;
    if (a->pair == GRAPE_CARRIED_FIRST && a->n_out % 2 != 0) return false;
    const uint32_t n = carried_pass_out(*a);
    return n >= a->period && n % a->period == 0 && a->n_out <= (1u << 30);
}
size_t grape_carried_partial_bytes(const grape_carried_args* args) {
    return carried_shape_ok(args) ? (size_t)carried_blocks(*args) * carried_values(*args) * 32 : 0;
}
int grape_carried_queue(const grape_carried_args* args, grape_stream_t st) {
    GRAPE_REQUIRE(carried_shape_ok(args) && args->pair == GRAPE_CARRIED_SINGLE, "n_out must be a whole number of periods, a period at most 2^20");
    const grape_carried_args& a = *args;
    CHECK_PTR16(a.A_out); CHECK_PTR16(a.Z_out); CHECK_PTR16(a.partial);
    hipStream_t s = as_stream(st);
    const uint32_t hstep = carried_step(a);
    const unsigned nb = carried_blocks(a);
    if (a.idx1) {
        CHECK_PTR16(a.halves); CHECK_PTR16(a.eq_high);
        GRAPE_REQUIRE(a.len >= 1, "empty table");
        carried_gather_kernel<<<nb, kBlock, 0, s>>>(a.A_out, a.Z_out, a.idx1, a.halves, a.len, a.eq_high, a.period, hstep, a.n_out, a.partial);
        GRAPE_LAUNCH_CHECK();
        return GRAPE_OK;
    }
    CHECK_PTR16(a.A); CHECK_PTR16(a.Z); CHECK_PTR16(a.eq);
    GRAPE_REQUIRE(a.tab_a != nullptr, "the round needs its challenge's table");
    if (a.eq_high) {
        CHECK_PTR16(a.eq_high);
        GRAPE_REQUIRE(!a.plain_sums, "the weights enter in a round without plain sums");
        carried_round_kernel<true, false><<<nb, kBlock, 0, s>>>(a.A_out, a.Z_out, a.A, a.Z, a.eq, a.eq_high, a.period, hstep, a.n_out, a.tab_a, nullptr, a.partial);
    } else {
        GRAPE_REQUIRE(a.tab_z != nullptr, "the round needs the carried tensor's table");
        if (a.plain_sums)
            carried_round_kernel<false, true><<<nb, kBlock, 0, s>>>(a.A_out, a.Z_out, a.A, a.Z, a.eq, nullptr, a.period, hstep, a.n_out, a.tab_a, a.tab_z, a.partial);
        else
            carried_round_kernel<false, false><<<nb, kBlock, 0, s>>>(a.A_out, a.Z_out, a.A, a.Z, a.eq, nullptr, a.period, hstep, a.n_out, a.tab_a, a.tab_z, a.partial);
    }
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
int grape_carried_queue_pair(const grape_carried_args* first, const grape_carried_args* second, grape_stream_t st) {
    GRAPE_REQUIRE(carried_shape_ok(first) && carried_shape_ok(second) && first->pair == GRAPE_CARRIED_FIRST && second->pair == GRAPE_CARRIED_SECOND,
                  "n_out must be a whole number of periods, a period at most 2^20");
    const grape_carried_args &a = *first, &b = *second;
    GRAPE_REQUIRE(a.n_out == 2 * b.n_out && a.period == b.period && a.eq == b.eq && !b.idx1 && !b.eq_high, "the second round follows the first one");
    CHECK_PTR16(b.A_out); CHECK_PTR16(b.Z_out); CHECK_PTR16(a.partial); CHECK_PTR16(b.partial); CHECK_PTR16(a.eq);
    GRAPE_REQUIRE(b.tab_a != nullptr && b.tab_z != nullptr, "the second round needs its tables");
    hipStream_t s = as_stream(st);
    const CarriedPair p{b.A_out, b.Z_out, a.A, a.Z, a.idx1, a.halves, a.len, a.eq, a.eq_high, a.period, carried_step(b), b.n_out,
                        a.tab_a, a.tab_z, b.tab_a, b.tab_z, a.partial, b.partial};
    const unsigned nb = carried_blocks(b);
    if (a.idx1) {
        CHECK_PTR16(a.halves); CHECK_PTR16(a.eq_high);
        GRAPE_REQUIRE(a.len >= 1, "empty table");
        GRAPE_REQUIRE(b.plain_sums, "a lookup's later rounds have plain sums");
        carried_pair_kernel<kGather, true><<<nb, kBlock, 0, s>>>(p);
        GRAPE_LAUNCH_CHECK();
        return GRAPE_OK;
    }
    CHECK_PTR16(a.A); CHECK_PTR16(a.Z);
    GRAPE_REQUIRE(a.tab_a != nullptr, "the round needs its challenge's table");
    GRAPE_REQUIRE(!a.plain_sums == !b.plain_sums, "rounds of one kind");
    if (a.eq_high) {
        CHECK_PTR16(a.eq_high);
        GRAPE_REQUIRE(!a.plain_sums, "the weights enter in a round without plain sums");
        carried_pair_kernel<kEnter, false><<<nb, kBlock, 0, s>>>(p);
    } else {
        GRAPE_REQUIRE(a.tab_z != nullptr, "the round needs the carried tensor's table");
        if (a.plain_sums) carried_pair_kernel<kLater, true><<<nb, kBlock, 0, s>>>(p);
        else carried_pair_kernel<kLater, false><<<nb, kBlock, 0, s>>>(p);
    }
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
int grape_carried_finish(uint32_t* sums, uint32_t stride, const grape_carried_args* rounds, uint32_t count, grape_stream_t st) {
    CHECK_PTR16(sums);
    GRAPE_REQUIRE(rounds != nullptr && count >= 1 && count <= kMaxCarried, "1..32 rounds");
    CarriedFinish f{};
    unsigned nb = 0;
    for (uint32_t i = 0; i < count; i++) {
        CHECK_PTR16(rounds[i].partial);
        GRAPE_REQUIRE(carried_shape_ok(&rounds[i]) && (rounds[i].idx1 != nullptr) == (rounds[0].idx1 != nullptr) && !rounds[i].plain_sums == !rounds[0].plain_sums,
                      "rounds of one kind");
        f.partial[i] = rounds[i].partial;
        f.nblocks[i] = carried_blocks(rounds[i]);
        f.out[i] = sums + (size_t)i * stride * 8;
        nb = nb > f.nblocks[i] ? nb : f.nblocks[i];
    }
    hipStream_t s = as_stream(st);
#define GRAPE_CFINAL(NV, NW)                                                                                   \
    do {                                                                                                       \
        if (nb >= kFinalWideMin) carried_final_kernel<NV, NW, kFinalBlock><<<count, kFinalBlock, 0, s>>>(f);   \
        else carried_final_kernel<NV, NW, kBlock><<<count, kBlock, 0, s>>>(f);                                 \
    } while (0)
    if (rounds[0].idx1) GRAPE_CFINAL(2, 0);
    else if (rounds[0].plain_sums) GRAPE_CFINAL(4, 2);
    else GRAPE_CFINAL(2, 2);
#undef GRAPE_CFINAL
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
int grape_carried_end(uint32_t* out, const uint32_t* Z, uint32_t n, const uint32_t* factor, uint32_t period, const uint32_t* beta, grape_stream_t st) {
    CHECK_PTR16(out); CHECK_PTR16(Z); CHECK_PTR16(factor);
    if (beta) CHECK_PTR16(beta);
    GRAPE_REQUIRE(n >= 1 && period >= 1, "nothing carried");
    carried_end_kernel<<<blocks_for(n), kBlock, 0, as_stream(st)>>>(out, Z, n, factor, period, beta);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

}  // extern "C"
