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
static uint32_t carried_hstep(const grape_carried_args& a) {
    const uint32_t periods = a.n_out / a.period;
    uint32_t hstep = (uint32_t)(kNumCU * 4 * kBlock) / a.period;
    if (hstep < 1) hstep = 1;
    while ((periods + hstep - 1) / hstep > kCarriedIters) hstep *= 2;
    return hstep < periods ? hstep : periods;
}
static unsigned carried_blocks(const grape_carried_args& a) { return blocks_for((size_t)carried_hstep(a) * a.period); }
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
    return a && a->period >= 1 && a->period <= GRAPE_WROUND_MAX_PERIOD && a->n_out >= a->period && a->n_out % a->period == 0 && a->n_out <= (1u << 30);
}
size_t grape_carried_partial_bytes(const grape_carried_args* args) {
    return carried_shape_ok(args) ? (size_t)carried_blocks(*args) * carried_values(*args) * 32 : 0;
}
int grape_carried_queue(const grape_carried_args* args, grape_stream_t st) {
    GRAPE_REQUIRE(carried_shape_ok(args), "n_out must be a whole number of periods, a period at most 2^20");
    const grape_carried_args& a = *args;
    CHECK_PTR16(a.A_out); CHECK_PTR16(a.Z_out); CHECK_PTR16(a.partial);
    hipStream_t s = as_stream(st);
    const uint32_t hstep = carried_hstep(a);
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
