// Sumcheck rounds whose terms carry an eq(u, x) weight: the element-product sumcheck (src/prove.cu:
// 119-172), phase 1 of the matmul sumcheck (:49-85), the claim-merging sumcheck (:245-300) and the
// logUp rounds of tLookup (src/tlookup.cu:117-244).  The reference materialises coefficient arrays
// and folds each of them over the remaining variables of u in every round; here a round is ONE
// pass over the operands: the weights come from a pyramid of eq tables built once per proof (no
// per-round halving), the operands are folded in place by the same pass, and the weighted sums
// leave the kernel as per-workgroup partial sums that a one-block kernel finishes.  Challenges are
// known before the first round, so the host queues all rounds and reads the sums once.
#include "fr_device.hpp"

namespace grape {

// ---------------------------------------------------------------- eq pyramid
// Level j (2^j entries) sits at element offset 2^j - 1; level j holds eq(u[0..j-1], i), bit b of i paired with u[b].
// Level by level (hi = lo * u[j], lo' = lo - hi) a pyramid is a chain of products, and above level 9 of launches, before a proof's
// first round.  Here levels up to kPyrTop are made at once, in one launch: a workgroup takes a head of 2^11 entries of a level that share their
// high bits, an entry is the product of a factor over bits 0..4, one over bits 5..10 and the head's own, and those are
// products of at most 6 (3 deep; 19 for the head, a tree over the lanes) factors u or 1 - u, made by different waves side by
// side.  One product an entry as before.  Bound by its chain of about 14 products below 2^16 entries, by issue above: 2^13 entries
// 26 -> 13 us and 5 -> 1 launches, 2^16 40 -> 13.5 and 8 -> 1.
// Up to kPyrShort variables an entry is its own product, three deep, and nothing meets anywhere: 3.8 to 6.2 us for 0 to 6 variables
// against 6.8 to 8.8 (7 variables 8.6 against 8.5 level by level).  Levels above kPyrTop are a launch each that reads the one
// below, half a product an entry: 21 variables 54 against 66 us, 22 90 against 124; one such level alone is not worth its launch
// (20 variables 38 against 41).
constexpr uint32_t kPyrLow = 5, kPyrHead = 11, kPyrShort = 6, kPyrTop = 19;

// the factor of u[b] for bit `set`; one for a variable that is not there
__device__ __forceinline__ Fr eq_factor(const uint32_t* u, uint32_t b, bool there, bool set) {
    if (!there) return Fr::one();
    const Fr x = ld_fr(u, b);
    return set ? x : sub(Fr::one(), x);
}
// the product of n <= 6 of them from u[b] on for the bits of i, three products deep
__device__ __forceinline__ Fr eq_factors(const uint32_t* u, uint32_t b, uint32_t n, uint32_t i) {
    Fr x[3];
#pragma unroll
    for (uint32_t k = 0; k < 3; k++)
        x[k] = fr26::mulc(eq_factor(u, b + 2 * k, 2 * k < n, (i >> 2 * k) & 1), eq_factor(u, b + 2 * k + 1, 2 * k + 1 < n, (i >> (2 * k + 1)) & 1));
    return fr26::mulc(fr26::mulc(x[0], x[1]), x[2]);
}
template <bool SHORT>
__global__ void __launch_bounds__(kBlock) eq_pyramid_head_kernel(uint32_t* pyr, const uint32_t* u, uint32_t nu) {
    if constexpr (SHORT) {
        // a thread an entry: entry i of a level is thread 2^level + i - 1
        const uint32_t at = threadIdx.x + 1, level = 31 - __clz(at), i = at - (1u << level);
        Fr f[kPyrShort];
#pragma unroll
        for (uint32_t j = 0; j < kPyrShort; j++)
            if (j < nu) f[j] = ld_fr(u, j);
        if (level > nu) return;
#pragma unroll
        for (uint32_t j = 0; j < kPyrShort; j++)
            if (j < nu) f[j] = j >= level ? Fr::one() : (i >> j) & 1 ? f[j] : sub(Fr::one(), f[j]);
        Fr x = nu > 1 ? fr26::mulc(f[0], f[1]) : nu ? f[0] : Fr::one();
        if (nu > 2) {
            Fr y = nu > 3 ? fr26::mulc(f[2], f[3]) : f[2];
            if (nu > 4) y = fr26::mulc(y, nu > 5 ? fr26::mulc(f[4], f[5]) : f[4]);
            x = fr26::mulc(x, y);
        }
        st_fr(pyr, threadIdx.x, x);
        return;
    }
    __shared__ Fr low[1 << kPyrLow], mid[1 << (kPyrHead - kPyrLow)], high;
    // workgroups 0..kPyrHead are the levels up to kPyrHead, 2^(level - kPyrHead) of them each level above
    uint32_t level = blockIdx.x, h = 0;
    if (level > kPyrHead) {
        const uint32_t i = blockIdx.x - kPyrHead + 1, lg = 31 - __clz(i);      // 2, 3 | 4, 5, 6, 7 | ...
        level = kPyrHead + lg;
        h = i - (1u << lg);
    }
    const uint32_t t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const uint32_t nlow = level < kPyrLow ? level : kPyrLow, nhead = level < kPyrHead ? level : kPyrHead, nmid = nhead - nlow;
    if (wave == 0) {
        if (lane < (1u << nlow)) low[lane] = eq_factors(u, 0, nlow, lane);
    } else if (wave == 1) {
        if (lane < (1u << nmid)) mid[lane] = eq_factors(u, nlow, nmid, lane);
    } else if (wave == 2) {
        const uint32_t rest = level - nhead;                // at most 19 of 32 lanes
        Fr x = eq_factor(u, kPyrHead + lane, lane < rest, (h >> (lane & 31)) & 1);
        for (uint32_t off = 16; off >= 1; off >>= 1) {
            if (off >= rest) continue;                      // the same for every lane
            const Fr y = shfl_down_fr(x, off);
            x = fr26::mulc(x, lane < off ? y : Fr::one());
        }
        if (lane == 0) high = x;
    }
    __syncthreads();
    if (wave == 1 && level > kPyrHead) mid[lane] = fr26::mulc(mid[lane], high);
    __syncthreads();
    const size_t at = ((size_t)1 << level) - 1 + ((size_t)h << kPyrHead);
    for (uint32_t i = t; i < (1u << nhead); i += kBlock) {
        const Fr l = low[i & ((1u << nlow) - 1)];
        st_fr(pyr, at + i, level > kPyrLow ? fr26::mulc(l, mid[i >> nlow]) : l);
    }
}

__global__ void __launch_bounds__(kBlock) eq_pyramid_level_kernel(uint32_t* pyr, const uint32_t* u, uint32_t j) {
    const size_t half = (size_t)1 << j, i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= half) return;
    const Fr lo = ld_fr(pyr, half - 1 + i), hi = fr26::mulc(lo, ld_fr(u, j));
    st_fr(pyr, 2 * half - 1 + half + i, hi);
    st_fr(pyr, 2 * half - 1 + i, sub(lo, hi));
}

// ---------------------------------------------------------------- weighted two-tensor round
// One thread runs at most kWIters indices; the three weighted sums are double-width column
// accumulators reduced once per thread.  Per index (e = weight, x0/x1 = halves of the MSB split,
// d = x1 - x0, S' = S + beta):
//   ea0 = e*a0 in (0, 1.46 r), ead = e*da in (0.54 r, 2.46 r)        (limbs normalised, below 2^26)
//   W0 += ea0 * s0'        < 2.92 r^2         s0' < 2r, limbs < 2^27
//   W2 += ead * ds         < 2.46 r^2         |ds| < r, |limb| < 2^26
//   WQ += (ea0+ead) * s1'  < 7.84 r^2         s1' < 2r, limbs < 2^27 -> a column grows by < 2^57.4
// so 24 indices keep a column below 2^62 and the sums within +-5.4 r of their offsets.  The sums
// leave the thread WITHOUT the radix factor 16 (value / 2^260, canonical); the finishing kernel
// applies it once.  The middle coefficient is WQ - W0 - W2 (one product instead of two).
constexpr int kWIters = 24;

// a finished column sum -> canonical element of value V / 2^260 + (a multiple of r)
__device__ __forceinline__ Fr reduce_to_fr(fr26::Acc& C, int lo_r) {
    return fr26::unpack(fr26::canon_wide(fr26::reduce(C, lo_r)));
}

// sums[0..2] = 16 * (W0, WQ - W0 - W2, W2); with PLAIN sums[3] = sum A0, sums[4] = sum A1 - sum A0
// UNIT (weights that sum to one, A * (S + beta) = 1 everywhere): sums[0] = 1, sums[1] = -sums[2]
// NOMID (the caller takes the middle coefficient from its running claim): sums[1] = 0
template <bool PLAIN, bool UNIT, bool NOMID>
__device__ __forceinline__ void wround2_result(uint32_t* out, const Fr* acc) {
    Fr w[3] = {acc[0], NOMID ? Fr::zero() : sub(sub(acc[1], acc[0]), acc[2]), acc[2]};
#pragma unroll
    for (int k = 0; k < 3; k++) {
        Fr t = w[k];
#pragma unroll
        for (int d = 0; d < 4; d++) t = add(t, t);
        w[k] = t;
    }
    if (UNIT) {
        w[0] = Fr::one();
        w[1] = sub(Fr::zero(), w[2]);
    }
#pragma unroll
    for (int k = 0; k < 3; k++) st_fr(out, k, w[k]);
    if (PLAIN) {
        st_fr(out, 3, acc[3]);
        st_fr(out, 4, sub(acc[4], acc[3]));
    }
}

// e * x reduced, add_r times r added.  TIGHT: as a plain sum (the five-sum form is at the limit of the registers).
template <bool TIGHT>
__device__ __forceinline__ fr26::Limbs weight_product(const fr26::Limbs& e16, const fr26::Limbs& x, int add_r) {
    if (!TIGHT) return fr26::product(e16, x, add_r);
    fr26::Acc T;
    fr26::acc_zero(T);
    fr26::mac(T, e16, x);
    return fr26::reduce(T, add_r);
}

// UNIT: the caller states that A[i] * (S[i] + beta) = 1 at every index (the first round of a logUp
// proof, where A was made as the inverse of S + beta).  Then the constant coefficient is the sum of
// the weights and the value at t = 1 equals it, so only the top coefficient sum_g e * dA * dS is
// taken: one weight product and one accumulation per index instead of two and three.
// TAB: the folds go through the table of the challenge's multiples (fr26::fold_table; long rounds).
// NOMID: the sum of the round polynomial over {0, 1} is known to the caller (the value the previous
// round's polynomial took at its challenge), which fixes the middle coefficient: the value at t = 1
// is not accumulated - one product and one double-width accumulator less per index.
// IDX: A is not read but gathered, A[i] = Bt[idx1[i] - 1] (in_size == 2 n_out): the first round of a lookup whose
// logUp tensor was never written out - the pass over the witness left the table indices only.  IDX = 2: nor is S, S[i] =
// Tt[idx1[i] - 1]; a witness element is read as its 4-byte index.  The tables' occupied entries sit in the caches (a
// softmax's in 64 KB), and what is saved is writing and reading both tensors: 2^27 elements, pass over the witness and first
// round 3.5 + 2.8 ms before.
// SPLIT: the weight of index h * period + l is Eh[h] * E[l].  A thread keeps one l, so E[l] is applied once, to its three sums,
// and what it reads per index is Eh[h] - the same word for a whole wave.  No table of n_out weights is made or read: building
// one and reading it back is 64 to 96 bytes an index pair beside the 192 of the operands (2^23 pairs and the levels below
// 2^20: 0.16 ms of launches, element product of 2048 x 11008: 0.30 ms).
template <bool BETA, bool PLAIN, bool UNIT, bool TAB, bool NOMID = false, int IDX = 0, bool SPLIT = false>
__global__ void __launch_bounds__(kBlock, 2) wround2_kernel(uint32_t* Aw, uint32_t* Sw, const uint32_t* A, const uint32_t* S,
                                                         const uint32_t* beta, const uint32_t* E,
                                                         uint32_t in_size, uint32_t n_out, uint32_t rowlen, uint32_t rowpad,
                                                         const uint32_t* v, const int32_t* __restrict__ tab, uint32_t* partial,
                                                         const int32_t* __restrict__ idx1 = nullptr, const uint32_t* Bt = nullptr,
                                                         const uint32_t* Eh = nullptr, uint32_t period = 1, const uint32_t* Tt = nullptr) {
    constexpr int NV = PLAIN ? 5 : 3;
    constexpr bool TIGHT = PLAIN && !UNIT && !NOMID;
    __shared__ Fr lds[NV * (kBlock / 64)];
    fr26::Limbs w1;
    if (!TAB) w1 = fr26::weight16(ld_fr(v, 0));
    fr26::Limbs bt;
    if (BETA) bt = fr26::pack(ld_fr(beta, 0));
    fr26::Acc W0, WQ, W2;
    fr26::acc_zero(W0);
    fr26::acc_zero(WQ);
    fr26::acc_zero(W2);
    fr26::Limbs sa0, sa1;                       // plain limb-wise sums of A's halves (24 terms below 2^26)
#pragma unroll
    for (int k = 0; k < fr26::N; k++) sa0.v[k] = sa1.v[k] = 0;
    size_t stride = (size_t)gridDim.x * kBlock;
    const size_t first = (size_t)blockIdx.x * kBlock + threadIdx.x;
    uint32_t h = 0, low = 0, hstep = 0;
    if (SPLIT) {
        hstep = (uint32_t)stride / period;
        stride = (size_t)hstep * period;             // whole periods: the threads behind them have no index
        h = (uint32_t)first / period;
        low = (uint32_t)first - h * period;
    }
    for (size_t g = SPLIT && first >= stride ? n_out : first; g < n_out; g += stride, h += hstep) {
        // weights live on rows of `rowpad` entries when the tensors' rows hold `rowlen` < rowpad
        const size_t ei = rowlen == rowpad ? g : g + (size_t)((uint32_t)g / rowlen) * (rowpad - rowlen);
        const fr26::Limbs e16 = fr26::pack16(SPLIT ? ld_fr(Eh, h) : ld_fr(E, ei));
        fr26::Limbs a0, a1;
        size_t t0 = 0, t1 = 0;
        if (IDX) {
            const uint32_t j0 = (uint32_t)idx1[g], j1 = (uint32_t)idx1[g + n_out];     // 0 marks an element outside the table
            t0 = j0 ? j0 - 1 : 0;
            t1 = j1 ? j1 - 1 : 0;
            a0 = ld_l26(Bt, t0);
            a1 = ld_l26(Bt, t1);
        } else {
            a0 = ld_l26(A, g);
            a1 = ld_hi26(A, g, n_out, in_size);
        }
        const fr26::Limbs da = fr26::sub(a1, a0);
        fr26::Limbs ea0;
        if (!UNIT) ea0 = weight_product<TIGHT>(e16, a0, 0);
        const fr26::Limbs ead = weight_product<TIGHT>(e16, da, 1);
        if (PLAIN) {
            sa0 = fr26::add(sa0, a0);
            sa1 = fr26::add(sa1, a1);
        }
        st_fr(Aw, g, TAB ? foldt1(tab, a0, da) : fold1(w1, a0, da));
        const fr26::Limbs s0r = IDX == 2 ? ld_l26(Tt, t0) : ld_l26(S, g);
        const fr26::Limbs s1r = IDX == 2 ? ld_l26(Tt, t1) : ld_hi26(S, g, n_out, in_size);
        const fr26::Limbs ds = fr26::sub(s1r, s0r);
        st_fr(Sw, g, TAB ? foldt1(tab, s0r, ds) : fold1(w1, s0r, ds));
        fr26::mac(W2, ead, ds);
        if (UNIT) {
            // W0 and WQ stay zero: the finishing kernel writes the coefficients they would give
        } else if (BETA) {
            fr26::mac(W0, ea0, fr26::add(s0r, bt));
            if (!NOMID) fr26::mac(WQ, fr26::add(ea0, ead), fr26::add(s1r, bt));
        } else {
            fr26::mac(W0, ea0, s0r);
            if (!NOMID) fr26::mac(WQ, fr26::add(ea0, ead), s1r);
        }
    }
    // offsets: |W0| < 71 r^2 -> within 2 r, |W2| < 60 r^2 -> within 1.7 r, |WQ| < 189 r^2 -> within 5.4 r
    Fr acc[NV];
    acc[0] = UNIT ? Fr::zero() : reduce_to_fr(W0, 3);
    acc[1] = UNIT || NOMID ? Fr::zero() : reduce_to_fr(WQ, 6);
    acc[2] = reduce_to_fr(W2, 3);
    if (SPLIT) {
        const Fr el = ld_fr(E, low);
        if (!UNIT) acc[0] = fr26::mulc(acc[0], el);
        if (!UNIT && !NOMID) acc[1] = fr26::mulc(acc[1], el);
        acc[2] = fr26::mulc(acc[2], el);
    }
    if (PLAIN) {
        acc[3] = fr26::limb_sum_to_fr(sa0, 0);      // below 24 r
        acc[4] = fr26::limb_sum_to_fr(sa1, 0);
    }
    block_sum<NV>(acc, lds);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < NV; k++) st_fr(partial, (size_t)blockIdx.x * NV + k, acc[k]);
    }
}
// One workgroup finishes one round; a proof that reads its sums at the end finishes all its long rounds in one launch.
constexpr uint32_t kMaxFinish = 32;
struct WFinish {
    const uint32_t* partial[kMaxFinish];
    uint32_t nblocks[kMaxFinish];
    uint32_t* out[kMaxFinish];
};
template <bool PLAIN, bool UNIT, bool NOMID, int BLOCK>
__global__ void __launch_bounds__(BLOCK) wround2_final_kernel(WFinish f) {
    constexpr int NV = PLAIN ? 5 : 3;
    __shared__ uint32_t lds9[NV * (BLOCK / 64) * 9];
    Fr tot[NV];
    workgroup_totals<NV, BLOCK, NOMID ? 2u : 0u>(tot, f.partial[blockIdx.x], f.nblocks[blockIdx.x], lds9);
    if (threadIdx.x == 0) wround2_result<PLAIN, UNIT, NOMID>(f.out[blockIdx.x], tot);
}

// ---------------------------------------------------------------- matmul phase 1: weights per segment
// Indices g = seg * seglen + k; every index of a segment shares the weight e[seg], so the three
// sums are taken per (segment, chunk) without weights and the finishing kernel applies e[seg].
__global__ void __launch_bounds__(kBlock) sumcheck2_seg_kernel(uint32_t* A, uint32_t* B, uint32_t in_size, uint32_t out_size,
                                                               uint32_t seglen, uint32_t seg0, const uint32_t* v, uint32_t* partial) {
    __shared__ Fr lds[3 * (kBlock / 64)];
    const fr26::Limbs w1 = fr26::weight16(ld_fr(v, 0));
    fr26::Acc C0, Q, C2;
    fr26::acc_zero(C0);
    fr26::acc_zero(Q);
    fr26::acc_zero(C2);
    const uint32_t seg = seg0 + blockIdx.y;            // a launch covers at most 65535 segments (the grid's y extent)
    const uint32_t stride = gridDim.x * kBlock;      // the host keeps seglen / stride <= 64
    for (uint32_t k = blockIdx.x * kBlock + threadIdx.x; k < seglen; k += stride) {
        const size_t g = (size_t)seg * seglen + k;
        if (g >= out_size) break;
        const fr26::Limbs a0 = ld_l26(A, g), b0 = ld_l26(B, g);
        const fr26::Limbs a1 = ld_hi26(A, g, out_size, in_size), b1 = ld_hi26(B, g, out_size, in_size);
        const fr26::Limbs da = fr26::sub(a1, a0), db = fr26::sub(b1, b0);
        st_fr(A, g, fold1(w1, a0, da));
        st_fr(B, g, fold1(w1, b0, db));
        fr26::mac(C0, a0, b0);
        fr26::mac(Q, a1, b1);
        fr26::mac(C2, da, db);
    }
    const Fr c0 = fr26::finish_sum(C0, 2), c2 = fr26::finish_sum(C2, 2), q1 = fr26::finish_sum(Q, 2);
    Fr acc[3] = {c0, sub(sub(q1, c0), c2), c2};
    block_sum<3>(acc, lds);
    if (threadIdx.x == 0) {
        const size_t slot = (size_t)seg * gridDim.x + blockIdx.x;
#pragma unroll
        for (int t = 0; t < 3; t++) st_fr(partial, slot * 3 + t, acc[t]);
    }
}
// sums[t] = sum_seg e[seg] * sum_chunk partial[seg][chunk][t]
__global__ void __launch_bounds__(kBlock) seg_final_kernel(uint32_t* out, const uint32_t* partial, const uint32_t* e, uint32_t nseg,
                                                           uint32_t nchunk) {
    __shared__ Fr lds[3 * (kBlock / 64)];
    Fr acc[3] = {Fr::zero(), Fr::zero(), Fr::zero()};
    for (uint32_t s = threadIdx.x; s < nseg; s += kBlock) {
        Fr t[3] = {Fr::zero(), Fr::zero(), Fr::zero()};
        for (uint32_t c = 0; c < nchunk; c++) {
#pragma unroll
            for (int k = 0; k < 3; k++) t[k] = add(t[k], ld_fr(partial, ((size_t)s * nchunk + c) * 3 + k));
        }
        const Fr w = ld_fr(e, s);
#pragma unroll
        for (int k = 0; k < 3; k++) acc[k] = add(acc[k], fr26::mulc(w, t[k]));
    }
    block_sum<3>(acc, lds);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < 3; k++) st_fr(out, k, acc[k]);
    }
}

// ---------------------------------------------------------------- claim merging: one tensor, several weight tables
// For claim j (blockIdx.y) with weights e_j: sums[2j] = sum_x e_j[x] X0[x], sums[2j+1] = sum_x e_j[x] (X1[x] - X0[x]).
// Nothing is modified (the fold is a separate launch: every claim reads the unfolded tensor).
struct PyrPack { const uint32_t* p[16]; };
__global__ void __launch_bounds__(kBlock) wsum1_kernel(const uint32_t* X, PyrPack E, uint32_t in_size, uint32_t n_out, uint32_t* partial) {
    __shared__ Fr lds[2 * (kBlock / 64)];
    const uint32_t* e = E.p[blockIdx.y];
    fr26::Acc C0, C1;
    fr26::acc_zero(C0);
    fr26::acc_zero(C1);
    const size_t stride = (size_t)gridDim.x * kBlock;
    // 64 indices per thread at most: e, x0 below 2^26 per limb -> a column grows by < 2^55.4 per index
    for (size_t g = (size_t)blockIdx.x * kBlock + threadIdx.x; g < n_out; g += stride) {
        const fr26::Limbs w = ld_l26(e, g);
        const fr26::Limbs x0 = ld_l26(X, g);
        const fr26::Limbs x1 = ld_hi26(X, g, n_out, in_size);
        fr26::mac(C0, w, x0);
        fr26::mac(C1, w, fr26::sub(x1, x0));
    }
    // |sum| < 64 r^2 -> within 1.82 r of the offset; the factor 16 is applied by the finishing kernel
    Fr acc[2] = {reduce_to_fr(C0, 2), reduce_to_fr(C1, 2)};
    block_sum<2>(acc, lds);
    if (threadIdx.x == 0) {
        const size_t slot = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
        st_fr(partial, slot * 2, acc[0]);
        st_fr(partial, slot * 2 + 1, acc[1]);
    }
}
__global__ void __launch_bounds__(kBlock) wsum1_final_kernel(uint32_t* out, const uint32_t* partial, uint32_t nblocks) {
    __shared__ Fr lds[2 * (kBlock / 64)];
    const uint32_t j = blockIdx.x;
    Fr acc[2] = {Fr::zero(), Fr::zero()};
    for (uint32_t b = threadIdx.x; b < nblocks; b += kBlock) {
        acc[0] = add(acc[0], ld_fr(partial, ((size_t)j * nblocks + b) * 2));
        acc[1] = add(acc[1], ld_fr(partial, ((size_t)j * nblocks + b) * 2 + 1));
    }
    block_sum<2>(acc, lds);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            Fr t = acc[k];
#pragma unroll
            for (int d = 0; d < 4; d++) t = add(t, t);
            st_fr(out, 2 * (size_t)j + k, t);
        }
    }
}

}  // namespace grape

using namespace grape;

extern "C" {

size_t grape_eq_pyramid_elems(uint32_t nu) { return ((size_t)2 << nu) - 1; }

int grape_eq_pyramid(uint32_t* pyr, const uint32_t* u, uint32_t nu, grape_stream_t st) {
    CHECK_PTR16(pyr);
    GRAPE_REQUIRE(nu <= 30, "too many variables");
    if (nu) CHECK_PTR16(u);
    hipStream_t s = as_stream(st);
    const uint32_t top = nu <= kPyrTop + 1 ? nu : kPyrTop;
    const unsigned nb = top <= kPyrHead ? top + 1 : kPyrHead - 1 + (1u << (top - kPyrHead + 1));
    if (nu <= kPyrShort) eq_pyramid_head_kernel<true><<<1, 2 << kPyrShort, 0, s>>>(pyr, u, nu);
    else eq_pyramid_head_kernel<false><<<nb, kBlock, 0, s>>>(pyr, u, top);
    for (uint32_t j = top; j < nu; j++) eq_pyramid_level_kernel<<<blocks_for((size_t)1 << j), kBlock, 0, s>>>(pyr, u, j);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

// workgroups of a weighted round over n_out index pairs
static unsigned wround2_blocks(uint32_t n_out) {
    unsigned nb = blocks_for(n_out);
    if (nb > (unsigned)kNumCU * 4) {
        const unsigned need = blocks_for(n_out, kBlock * kWIters);
        nb = need > (unsigned)kNumCU * 4 ? need : (unsigned)kNumCU * 4;
    }
    return nb;
}

// The two launches of a weighted round: the pass over the operands (partial sums per workgroup; `tab`: the table of
// the challenge's multiples, or nullptr for the single-product fold) and the kernel that finishes the sums.
// The folded operands go to Aw and Sw (A and S themselves for a round in place).
static int wround2_main(uint32_t* Aw, uint32_t* Sw, const uint32_t* A, const uint32_t* S, const uint32_t* beta, const uint32_t* E, uint32_t in_size, uint32_t n_out,
                        uint32_t rowlen, uint32_t rowpad, const uint32_t* v, int plain_sums, const int32_t* tab, uint32_t* partial,
                        hipStream_t s) {
    const unsigned nb = wround2_blocks(n_out);
    const bool use_tab = tab != nullptr;
    // five sums and three accumulators leave no registers for the table fold's columns (it spills: 1.16 against
    // 1.10 ms at 2^24 index pairs), so that form keeps the single-product fold at every size
#define GRAPE_WROUND2(B, P, U)                                                                                        \
    do {                                                                                                              \
        if (use_tab && !((P) && !(U)))                                                                                \
            wround2_kernel<B, P, U, !((P) && !(U))><<<nb, kBlock, 0, s>>>(Aw, Sw, A, S, beta, E, in_size, n_out, rowlen, rowpad, v, tab, partial); \
        else wround2_kernel<B, P, U, false><<<nb, kBlock, 0, s>>>(Aw, Sw, A, S, beta, E, in_size, n_out, rowlen, rowpad, v, nullptr, partial);    \
    } while (0)
    if (plain_sums == 3) {
        // the middle coefficient is left to the caller (sums[1] = 0); long rounds of a logUp proof
        GRAPE_REQUIRE(beta != nullptr && use_tab, "the round without its middle coefficient is built for logUp rounds of 2^16 index pairs and more");
        wround2_kernel<true, true, false, true, true><<<nb, kBlock, 0, s>>>(Aw, Sw, A, S, beta, E, in_size, n_out, rowlen, rowpad, v, tab, partial);
    } else if (plain_sums == 2) {
        GRAPE_REQUIRE(rowlen == rowpad && in_size == 2 * (uint64_t)n_out,
                      "the inverse-pair round needs whole pairs and unpadded rows (weights that sum to one)");
        if (beta) GRAPE_WROUND2(true, true, true);
        else GRAPE_WROUND2(false, true, true);
    } else if (beta && plain_sums) {
        GRAPE_WROUND2(true, true, false);
    } else if (beta) {
        GRAPE_WROUND2(true, false, false);
    } else if (plain_sums) {
        GRAPE_WROUND2(false, true, false);
    } else {
        GRAPE_WROUND2(false, false, false);
    }
#undef GRAPE_WROUND2
    return GRAPE_OK;
}
static void wround2_final(const WFinish& f, uint32_t count, int plain_sums, hipStream_t s) {
    unsigned nb = 0;
    for (uint32_t i = 0; i < count; i++) nb = std::max(nb, f.nblocks[i]);
#define GRAPE_WFINAL(P, U, M)                                                                            \
    do {                                                                                                 \
        if (nb >= kFinalWideMin) wround2_final_kernel<P, U, M, kFinalBlock><<<count, kFinalBlock, 0, s>>>(f); \
        else wround2_final_kernel<P, U, M, kBlock><<<count, kBlock, 0, s>>>(f);                          \
    } while (0)
    if (plain_sums == 3) GRAPE_WFINAL(true, false, true);
    else if (plain_sums == 2) GRAPE_WFINAL(true, true, false);
    else if (plain_sums) GRAPE_WFINAL(true, false, false);
    else GRAPE_WFINAL(false, false, false);
#undef GRAPE_WFINAL
}
// workgroups of a round with split weights: a power of two, so that 256 CUs with two workgroups each are filled evenly, and
// enough of them for at most kWIters whole periods per thread
static unsigned wround_split_blocks(uint32_t n_out, uint32_t period) {
    const uint64_t periods = ((uint64_t)n_out + period - 1) / period;
    unsigned nb = kNumCU * 4;
    while (true) {
        const uint64_t step = (uint64_t)nb * kBlock / period;
        if (step && (periods + step - 1) / step <= kWIters) return nb;
        nb *= 2;
    }
}
static unsigned wround_blocks(const grape_wround_args& a) { return a.eq_high ? wround_split_blocks(a.n_out, a.period) : wround2_blocks(a.n_out); }
#define GRAPE_WROUND2_CHECKS()                                                                                              \
    CHECK_PTR16(A); CHECK_PTR16(S); CHECK_PTR16(E); CHECK_PTR16(v);                                                        \
    GRAPE_REQUIRE(n_out >= 1 && in_size >= n_out && in_size <= 2 * (uint64_t)n_out, "need n_out <= in_size <= 2*n_out"); \
    GRAPE_REQUIRE(rowlen >= 1 && rowlen <= rowpad, "need 1 <= rowlen <= rowpad");                                        \
    if (beta) CHECK_PTR16(beta)

// The round as a value: what grape_wround_queue and grape_wround_finish take (folded in place, one table of weights).
static grape_wround_args wround2_args(uint32_t* A, uint32_t* S, const uint32_t* beta, const uint32_t* E, uint32_t in_size, uint32_t n_out, uint32_t rowlen,
                                      uint32_t rowpad, const uint32_t* v, int plain_sums, const int32_t* tab, uint32_t* partial) {
    grape_wround_args a{};
    a.A = a.A_out = A;
    a.S = a.S_out = S;
    a.beta = beta;
    a.eq = E;
    a.rowlen = rowlen;
    a.rowpad = rowpad;
    a.in_size = in_size;
    a.n_out = n_out;
    a.v = v;
    a.plain_sums = plain_sums;
    a.tab = tab;
    a.partial = partial;
    return a;
}
int grape_wround2(uint32_t* A, uint32_t* S, const uint32_t* beta, const uint32_t* E, uint32_t in_size, uint32_t n_out,
                  uint32_t rowlen, uint32_t rowpad, const uint32_t* v, int plain_sums, uint32_t* sums, grape_stream_t st) {
    GRAPE_WROUND2_CHECKS();
    CHECK_PTR16(sums);
    hipStream_t s = as_stream(st);
    void* ws;
    const size_t partial_bytes = (size_t)wround2_blocks(n_out) * (plain_sums ? 5 : 3) * 32;
    int rc = scratch_get(kSlotReduce, partial_bytes + kFoldTableBytes, &ws, s);
    if (rc) return rc;
    // long rounds fold through the table of the challenge's multiples (one more small launch)
    int32_t* tab = nullptr;
    if (n_out >= kTableFoldMinOut) {
        tab = (int32_t*)((char*)ws + partial_bytes);
        fold_tables_kernel<<<1, 64, 0, s>>>(tab, v, 1);
    }
    const grape_wround_args a = wround2_args(A, S, beta, E, in_size, n_out, rowlen, rowpad, v, plain_sums, tab, (uint32_t*)ws);
    rc = grape_wround_queue(&a, st);
    return rc ? rc : grape_wround_finish(sums, 0, &a, 1, st);
}

size_t grape_wround2_partial_bytes(uint32_t n_out) { return (size_t)wround2_blocks(n_out ? n_out : 1) * 5 * 32; }

static_assert(GRAPE_FOLD_TABLE_WORDS == fr26::kFoldTableWords, "the header's table size is the kernels'");
int grape_fold_tables(int32_t* tabs, const uint32_t* v, uint32_t count, grape_stream_t st) {
    GRAPE_REQUIRE(tabs != nullptr && (reinterpret_cast<uintptr_t>(tabs) & 3) == 0, "tabs must be 4-byte aligned");
    GRAPE_REQUIRE(count >= 1 && count <= 64, "1..64 challenges");
    CHECK_PTR16(v);
    fold_tables_kernel<<<count, 64, 0, as_stream(st)>>>(tabs, v, count);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

int grape_wround2_queue(uint32_t* A, uint32_t* S, const uint32_t* beta, const uint32_t* E, uint32_t in_size, uint32_t n_out,
                        uint32_t rowlen, uint32_t rowpad, const uint32_t* v, int plain_sums, const int32_t* tab, uint32_t* partial,
                        grape_stream_t st) {
    const grape_wround_args a = wround2_args(A, S, beta, E, in_size, n_out, rowlen, rowpad, v, plain_sums, tab, partial);
    return grape_wround_queue(&a, st);
}

int grape_wround2_queue_indexed(uint32_t* A, uint32_t* S, const int32_t* idx1, const uint32_t* Bt, uint32_t len, const uint32_t* beta,
                                const uint32_t* E, uint32_t n_out, const uint32_t* v, const int32_t* tab, uint32_t* partial,
                                grape_stream_t st) {
    GRAPE_REQUIRE(idx1 != nullptr && len >= 1 && n_out <= (1u << 30), "bad arguments");
    grape_wround_args a = wround2_args(A, S, beta, E, 2 * n_out, n_out, 1, 1, v, 2, tab, partial);
    a.idx1 = idx1;
    a.B = Bt;
    return grape_wround_queue(&a, st);
}

size_t grape_wround_partial_bytes(const grape_wround_args* args) {
    if (!args || args->n_out < 1 || (args->eq_high && (args->period < 1 || args->period > GRAPE_WROUND_MAX_PERIOD))) return 0;
    return (size_t)wround_blocks(*args) * (args->plain_sums ? 5 : 3) * 32;
}
// T: with idx1, S is gathered from it too
static int wround_queue_impl(const grape_wround_args* args, const uint32_t* T, grape_stream_t st) {
    GRAPE_REQUIRE(args != nullptr, "null arguments");
    const grape_wround_args& a = *args;
    const uint32_t *A = T ? T : a.A, *S = T ? T : a.S, *E = a.eq, *v = a.v, *beta = a.beta;     // neither is read with T
    const uint32_t in_size = a.in_size, n_out = a.n_out, rowlen = a.rowlen, rowpad = a.rowpad;
    GRAPE_WROUND2_CHECKS();
    CHECK_PTR16(a.A_out); CHECK_PTR16(a.S_out); CHECK_PTR16(a.partial);
    hipStream_t s = as_stream(st);
    const unsigned nb = wround_blocks(a);
    GRAPE_REQUIRE(a.tab == nullptr || n_out >= kTableFoldMinOut, "the table fold is built for rounds of 2^16 index pairs and more");
    GRAPE_REQUIRE((a.idx1 == nullptr && a.eq_high == nullptr) || a.tab != nullptr, "indexed rounds and split weights need the challenge's table");
    if (a.idx1) {
        CHECK_PTR16(a.B);
        GRAPE_REQUIRE(a.plain_sums == 2 && beta && in_size == 2 * (uint64_t)n_out && rowlen == rowpad, "an indexed round is a lookup's first round");
    }
    if (!a.eq_high) {
        if (a.idx1 && T)
            wround2_kernel<true, true, true, true, false, 2><<<nb, kBlock, 0, s>>>(a.A_out, a.S_out, A, S, beta, E, in_size, n_out, 1, 1, v, a.tab,
                                                                                  a.partial, a.idx1, a.B, nullptr, 1, T);
        else if (a.idx1)
            wround2_kernel<true, true, true, true, false, 1><<<nb, kBlock, 0, s>>>(a.A_out, a.S_out, A, S, beta, E, in_size, n_out, 1, 1, v, a.tab,
                                                                                  a.partial, a.idx1, a.B);
        else if (int rc = wround2_main(a.A_out, a.S_out, A, S, beta, E, in_size, n_out, rowlen, rowpad, v, a.plain_sums, a.tab, a.partial, s)) return rc;
        GRAPE_LAUNCH_CHECK();
        return GRAPE_OK;
    }
    CHECK_PTR16(a.eq_high);
    GRAPE_REQUIRE(a.period >= 1 && a.period <= GRAPE_WROUND_MAX_PERIOD, "the period of split weights is 1..2^20");
#define GRAPE_WSPLIT(BETA, P, U, M, I)                                                                                           \
    wround2_kernel<BETA, P, U, true, M, I, true><<<nb, kBlock, 0, s>>>(a.A_out, a.S_out, A, S, beta, E, in_size, n_out, 1, 1, v, a.tab, \
                                                                    a.partial, a.idx1, a.B, a.eq_high, a.period, T)
    if (a.plain_sums == 0 && !beta) GRAPE_WSPLIT(false, false, false, false, 0);
    else if (a.plain_sums == 3 && beta) GRAPE_WSPLIT(true, true, false, true, 0);
    else if (a.plain_sums == 2 && beta && a.idx1 && T) GRAPE_WSPLIT(true, true, true, false, 2);
    else if (a.plain_sums == 2 && beta && a.idx1) GRAPE_WSPLIT(true, true, true, false, 1);
    else if (a.plain_sums == 2 && beta && in_size == 2 * (uint64_t)n_out) GRAPE_WSPLIT(true, true, true, false, 0);
    else GRAPE_REQUIRE(false, "split weights are built for plain_sums 0 without beta and for 2 and 3 with it");
#undef GRAPE_WSPLIT
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
int grape_wround_queue(const grape_wround_args* args, grape_stream_t st) { return wround_queue_impl(args, nullptr, st); }
int grape_wround_queue_gathered(const grape_wround_args* args, const uint32_t* T, grape_stream_t st) {
    CHECK_PTR16(T);
    GRAPE_REQUIRE(args != nullptr && args->idx1 != nullptr, "a gathered round needs the table indices");
    return wround_queue_impl(args, T, st);
}
int grape_wround_finish(uint32_t* sums, uint32_t stride, const grape_wround_args* rounds, uint32_t count, grape_stream_t st) {
    CHECK_PTR16(sums);
    GRAPE_REQUIRE(rounds != nullptr && count >= 1 && count <= kMaxFinish, "1..32 rounds");
    WFinish f{};
    for (uint32_t i = 0; i < count; i++) {
        CHECK_PTR16(rounds[i].partial);
        GRAPE_REQUIRE(rounds[i].plain_sums == rounds[0].plain_sums && grape_wround_partial_bytes(&rounds[i]) != 0, "rounds of one kind");
        f.partial[i] = rounds[i].partial;
        f.nblocks[i] = wround_blocks(rounds[i]);
        f.out[i] = sums + (size_t)i * stride * 8;
    }
    wround2_final(f, count, rounds[0].plain_sums, as_stream(st));
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

int grape_wround2_finish(uint32_t* sums, const uint32_t* partial, uint32_t n_out, int plain_sums, grape_stream_t st) {
    grape_wround_args a{};
    a.n_out = n_out;
    a.plain_sums = plain_sums;
    a.partial = const_cast<uint32_t*>(partial);
    return grape_wround_finish(sums, 0, &a, 1, st);
}
#undef GRAPE_WROUND2_CHECKS

int grape_sumcheck_round2_seg(uint32_t* A, uint32_t* B, uint32_t in_size, uint32_t out_size, uint32_t seglen, const uint32_t* e,
                              const uint32_t* v, uint32_t* sums, grape_stream_t st) {
    CHECK_PTR16(A); CHECK_PTR16(B); CHECK_PTR16(e); CHECK_PTR16(v); CHECK_PTR16(sums);
    GRAPE_REQUIRE(out_size >= 1 && in_size >= out_size && in_size <= 2 * (uint64_t)out_size, "need out_size <= in_size <= 2*out_size");
    GRAPE_REQUIRE(seglen >= 1 && out_size % seglen == 0, "out_size must be a whole number of segments");
    const uint32_t nseg = out_size / seglen;
    hipStream_t s = as_stream(st);
    // chunks per segment: one index per thread until the grid is large, never more than 64 per thread
    uint32_t nchunk = blocks_for(seglen);
    const uint32_t cap = nseg >= 2048 ? 1 : 2048 / nseg;
    if (nchunk > cap) nchunk = cap;
    const uint32_t need = blocks_for(seglen, kBlock * 64);
    if (nchunk < need) nchunk = need;
    void* ws;
    int rc = scratch_get(kSlotReduce, (size_t)nseg * nchunk * 3 * 32, &ws, s);
    if (rc) return rc;
    for (uint32_t seg0 = 0; seg0 < nseg; seg0 += 65535) {
        const uint32_t ns = nseg - seg0 < 65535 ? nseg - seg0 : 65535;
        sumcheck2_seg_kernel<<<dim3(nchunk, ns), kBlock, 0, s>>>(A, B, in_size, out_size, seglen, seg0, v, (uint32_t*)ws);
    }
    seg_final_kernel<<<1, kBlock, 0, s>>>(sums, (const uint32_t*)ws, e, nseg, nchunk);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

int grape_wsum1_multi(const uint32_t* X, const uint32_t* const* e_tables, uint32_t num, uint32_t in_size, uint32_t n_out,
                      uint32_t* sums, grape_stream_t st) {
    CHECK_PTR16(X); CHECK_PTR16(sums);
    GRAPE_REQUIRE(e_tables != nullptr && num >= 1 && num <= 16, "1..16 weight tables");
    GRAPE_REQUIRE(n_out >= 1 && in_size >= n_out && in_size <= 2 * (uint64_t)n_out, "need n_out <= in_size <= 2*n_out");
    PyrPack pk;
    for (uint32_t j = 0; j < 16; j++) pk.p[j] = j < num ? e_tables[j] : nullptr;
    for (uint32_t j = 0; j < num; j++) CHECK_PTR16(pk.p[j]);
    hipStream_t s = as_stream(st);
    unsigned nb = blocks_for(n_out);
    if (nb > (unsigned)kNumCU * 4) {
        const unsigned need = blocks_for(n_out, kBlock * 64);
        nb = need > (unsigned)kNumCU * 4 ? need : (unsigned)kNumCU * 4;
    }
    void* ws;
    int rc = scratch_get(kSlotReduce, (size_t)nb * num * 2 * 32, &ws, s);
    if (rc) return rc;
    wsum1_kernel<<<dim3(nb, num), kBlock, 0, s>>>(X, pk, in_size, n_out, (uint32_t*)ws);
    wsum1_final_kernel<<<num, kBlock, 0, s>>>(sums, (const uint32_t*)ws, nb);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

}  // extern "C"
