// The short rounds of a sumcheck - all rounds that are left once a tensor holds at most 2^17 elements - in four or five
// launches instead of two a round.  (2^17: longer rounds fold through the challenge's table and are bound by their work.)
//
// A short round moves a few KB to a few MB: it is bound by latency (a chain of three or four dependent field products, a
// workgroup sum, a launch, a finishing launch), not by work, and a proof has 10 to 17 of them on every chain.  The
// challenges of a proof are known before its first round, so nothing but the FOLDS is a chain: folding is one
// product, and the sums of all rounds can be taken side by side once the folded tensors are there.  So
//   fold_levels_kernel   folds nine variables a launch: a workgroup loads the 512 elements whose indices agree in the
//                        low bits (an MSB fold pairs i with i + n/2, so they fold onto each other), folds them in LDS and writes
//                        EVERY level to memory; one tensor per grid row;
//   round_sums_kernel    takes the sums of all rounds at once, one wave per (64 index pairs, product): the products of a
//                        pair are spread over waves, and a wave's sum is limb-wise adds along a row of lanes;
//   round_finish_kernel  adds up the partial sums, one workgroup per round.
// A range lookup of 2^14 elements: 0.81 -> 0.44 ms; a matmul proof over 32 heads (12 rounds): 0.39 -> 0.18 ms.
#include "fr_device.hpp"

namespace grape {

constexpr uint32_t kShortMaxElems = 1u << 17;
constexpr uint32_t kShortMaxRounds = 17;
constexpr int kLevelElems = 512;          // elements of one workgroup of fold_levels_kernel
constexpr uint32_t kLevelVars = 9;

struct FoldSeg {
    const uint32_t* src[3];
    uint32_t* lev[3];                      // level buffers; element offset off[t] starts the tensor after t rounds
    const uint32_t* v_end;                 // round t binds v_end[-(t+1)]
    uint32_t live, stride, k, cshift, t0;  // live elements of src, its residues mod `stride`, variables folded here, first round
    uint32_t off[kShortMaxRounds + 1];
};

// Bound by latency: `k` times (one product, one barrier).  Two elements a thread at the first level; the levels stay in LDS
// word by word (lane stride one word).
__global__ void __launch_bounds__(kBlock) fold_levels_kernel(FoldSeg s) {
    __shared__ uint32_t el[8][kLevelElems];
    __shared__ fr26::Limbs w[kLevelVars];
    const uint32_t* src = s.src[blockIdx.y];
    uint32_t* lev = s.lev[blockIdx.y];
    const uint32_t c = 1u << s.cshift, r0 = blockIdx.x << s.cshift, n = 1u << (s.k + s.cshift);
    for (uint32_t i = threadIdx.x; i < n; i += kBlock) {
        const uint32_t r = r0 + (i & (c - 1)), g = (i >> s.cshift) * s.stride + r;
        const Fr x = r < s.stride && g < s.live ? ld_fr(src, g) : Fr::zero();
#pragma unroll
        for (int q = 0; q < 8; q++) el[q][i] = x.v[q];
    }
    if (threadIdx.x >= kBlock - 64 && threadIdx.x - (kBlock - 64) < s.k) {
        const uint32_t t = threadIdx.x - (kBlock - 64);
        w[t] = fr26::weight16(ld_fr(s.v_end - 8 * (size_t)(s.t0 + t + 1), 0));
    }
    __syncthreads();
    for (uint32_t t = 0; t < s.k; t++) {
        const uint32_t half = n >> (t + 1), i = threadIdx.x;
        if (i < half) {
            Fr lo, hi;
#pragma unroll
            for (int q = 0; q < 8; q++) {
                lo.v[q] = el[q][i];
                hi.v[q] = el[q][i + half];
            }
            const fr26::Limbs l = fr26::pack(lo);
            const Fr x = fold1(w[t], l, fr26::sub(fr26::pack(hi), l));
#pragma unroll
            for (int q = 0; q < 8; q++) el[q][i] = x.v[q];
            const uint32_t r = r0 + (i & (c - 1));
            if (r < s.stride) st_fr(lev, s.off[s.t0 + t + 1] + (size_t)(i >> s.cshift) * s.stride + r, x);
        }
        __syncthreads();
    }
}

struct RoundSums {
    const uint32_t* x[3];
    const uint32_t* lev[3];
    const uint32_t *beta, *pyramid;
    uint32_t* partial;
    uint32_t rounds, top_level;
    uint32_t chunk0[kShortMaxRounds + 1], in[kShortMaxRounds], out[kShortMaxRounds], off[kShortMaxRounds + 1];
    // weights of a round: none (rowlen 0), entry g / rowlen (rowpad 0), or entry g of rows padded from rowlen to rowpad
    uint32_t rowlen[kShortMaxRounds], rowpad[kShortMaxRounds];
};

// sum over the wave of limbs whose 16-lane sums lie in (-add_r r, (32 - add_r) r); the same in every lane
__device__ __forceinline__ Fr wave_limb_sum(const fr26::Limbs& a, int add_r) {
    const Fr f = fr26::limb_sum_to_fr(row_sum(a), add_r);
    Fr q[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
#pragma unroll
        for (int i = 0; i < 8; i++) q[r].v[i] = (uint32_t)__builtin_amdgcn_readlane((int)f.v[i], 16 * r + 15);
    }
    return add(add(q[0], q[1]), add(q[2], q[3]));
}

// Wave q of a workgroup takes product q of 64 index pairs.  With x, y the halves of two tensors (y' = y + beta):
//   q = 0: x0 y0'    q = 1: x1 y1'    q = 2: (x1 - x0)(y1 - y0)        each times the pair's weight
// PLAIN: waves 0 and 1 also add up x0 and x1.  TABLE: (x, y) = (tensor 0, tensor 1) in waves 0 to 2 and, with neither beta
// nor weights, (tensor 2, tensor 0) in waves 3 to 5.
// Bounds (r / 2^260 = 1/35.3): x y' < 2 r^2 leaves the first reduction in (0, 1.91 r), the signed product in (-0.46 r, 1.46 r);
// the weight's product is in (0, 1.87 r) resp. (-0.21 r, 1.67 r): sixteen of them within (-4 r, 30 r), and sixteen unweighted
// ones within (0, 23.4 r) (no beta there) resp. (-8 r, 23.4 r).
template <bool PLAIN, bool TABLE>
__global__ void __launch_bounds__(64 * (TABLE ? 6 : 3)) round_sums_kernel(RoundSums a) {
    constexpr int NV = TABLE ? 8 : PLAIN ? 5 : 3;
    const int q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kind = q % 3;
    const bool mb = q >= 3;
    uint32_t t = 0;
    while (t + 1 < a.rounds && blockIdx.x >= a.chunk0[t + 1]) t++;
    const uint32_t g = (blockIdx.x - a.chunk0[t]) * 64 + (threadIdx.x & 63), out = a.out[t], in = a.in[t];
    const int ix = mb ? 2 : 0, iy = mb ? 0 : 1;
    const uint32_t* X = t ? a.lev[ix] + 8 * (size_t)a.off[t] : a.x[ix];
    const uint32_t* Y = t ? a.lev[iy] + 8 * (size_t)a.off[t] : a.x[iy];
    const bool live = g < out, weighted = !mb && a.rowlen[t] != 0;
    Fr x = Fr::zero(), y = Fr::zero(), x1 = Fr::zero(), y1 = Fr::zero(), e = Fr::zero();
    if (live) {
        if (kind != 1) {
            x = ld_fr(X, g);
            y = ld_fr(Y, g);
        }
        if (kind != 0) {
            x1 = ld_hi(X, g, out, in);
            y1 = ld_hi(Y, g, out, in);
        }
        if (weighted) {
            const uint32_t row = g / a.rowlen[t];
            const uint32_t i = a.rowpad[t] ? g + row * (a.rowpad[t] - a.rowlen[t]) : row;
            e = ld_fr(a.pyramid, ((size_t)1 << (a.top_level - t)) - 1 + i);
        }
    }
    fr26::Limbs l = fr26::pack(kind == 1 ? x1 : x), m = fr26::pack(kind == 1 ? y1 : y);
    const fr26::Limbs plain = l;
    if (kind == 2) {
        l = fr26::sub(fr26::pack(x1), l);
        m = fr26::sub(fr26::pack(y1), m);
    } else if (!mb && a.beta) {
        m = fr26::add(m, fr26::pack(ld_fr(a.beta, 0)));
    }
#pragma unroll
    for (int i = 0; i < fr26::N; i++) l.v[i] *= 16;
    fr26::Limbs p = fr26::product(l, m, 0);
    if (weighted) p = fr26::product(fr26::pack16(e), p, 0);
    const Fr sum = wave_limb_sum(p, kind != 2 ? 0 : weighted ? 4 : 8);
    uint32_t* slot = a.partial + 8 * (size_t)NV * blockIdx.x;
    if ((threadIdx.x & 63) == 0) st_fr(slot, mb ? q + 2 : q, sum);
    if (PLAIN && q < 2) {
        const Fr s = wave_limb_sum(plain, 0);
        if ((threadIdx.x & 63) == 0) st_fr(slot, 3 + q, s);
    }
}

struct RoundFinish {
    const uint32_t* partial;
    uint32_t* sums;
    uint32_t stride, rounds;               // sums of round t at element t * stride
    uint32_t chunk0[kShortMaxRounds + 1];
    const uint32_t* end[3];                // the element that is left of each tensor
    uint32_t *last[3], *copy[3];
};
template <int NV>
__global__ void __launch_bounds__(kBlock) round_finish_kernel(RoundFinish a) {
    __shared__ uint32_t lds9[NV * (kBlock / 64) * 9];
    const uint32_t t = blockIdx.x;
    if (t == a.rounds) {
        if (threadIdx.x < 8) {
            for (int k = 0; k < 3; k++) {
                if (!a.end[k]) continue;
                const uint32_t x = a.end[k][threadIdx.x];
                if (a.last[k]) a.last[k][threadIdx.x] = x;
                if (a.copy[k]) a.copy[k][threadIdx.x] = x;
            }
        }
        return;
    }
    Fr s[NV];
    workgroup_totals<NV, kBlock>(s, a.partial + 8 * (size_t)NV * a.chunk0[t], a.chunk0[t + 1] - a.chunk0[t], lds9);
    if (threadIdx.x != 0) return;
    // values at 0 and 1 and the top coefficient: the middle one is the value at 1 less the two others
    s[1] = sub(sub(s[1], s[0]), s[2]);
    if (NV >= 5) s[4] = sub(s[4], s[3]);
    if (NV == 8) s[6] = sub(sub(s[6], s[5]), s[7]);
#pragma unroll
    for (int k = 0; k < NV; k++) st_fr(a.sums, (size_t)t * a.stride + k, s[k]);
}

static uint32_t log2_ceil(uint32_t n) {
    uint32_t l = 0;
    while (((uint64_t)1 << l) < n) l++;
    return l;
}

}  // namespace grape

using namespace grape;

extern "C" int grape_short_rounds(const struct grape_short_rounds_args* p, grape_stream_t st) {
    GRAPE_REQUIRE(p != nullptr, "null arguments");
    const bool logup = p->kind == GRAPE_SHORT_LOGUP, table = p->kind == GRAPE_SHORT_TABLE;
    GRAPE_REQUIRE(p->kind == GRAPE_SHORT_PAIR || logup || table, "unknown kind of rounds");
    GRAPE_REQUIRE(p->size >= 2 && p->size <= kShortMaxElems, "2 to 2^17 elements");
    GRAPE_REQUIRE(p->row >= 1 && p->row <= p->size && p->size % p->row == 0, "the tensors must hold whole rows");
    const uint32_t nrows = p->size / p->row;
    GRAPE_REQUIRE((nrows & (nrows - 1)) == 0, "the number of rows must be a power of two");
    const int nt = table ? 3 : 2, NV = table ? 8 : logup ? 5 : 3;
    for (int k = 0; k < nt; k++) CHECK_PTR16(p->x[k]);
    CHECK_PTR16(p->v_end); CHECK_PTR16(p->sums);
    for (int k = 0; k < nt; k++) {
        if (p->last[k]) CHECK_PTR16(p->last[k]);
        if (p->last_copy[k]) CHECK_PTR16(p->last_copy[k]);
    }
    GRAPE_REQUIRE(p->weights <= GRAPE_SHORT_ROWS && (p->weights == GRAPE_SHORT_FULL || !(logup || table)), "lookup rounds weigh every index");
    if (p->weights) CHECK_PTR16(p->pyramid);
    if (p->beta) CHECK_PTR16(p->beta);
    GRAPE_REQUIRE(p->beta == nullptr || p->weights == GRAPE_SHORT_FULL, "a shift needs weighted rounds");
    const uint32_t rows_log = log2_ceil(nrows), row_log = log2_ceil(p->row), rounds = rows_log + row_log;
    GRAPE_REQUIRE(rounds >= 1 && rounds <= kShortMaxRounds && p->stride >= (uint32_t)NV, "bad arguments");

    // what every round reads and leaves: whole rows are paired until one is left, which is taken as padded with zeros
    RoundSums rs = {};
    uint32_t in = p->size, chunks = 0;
    size_t total = 0;
    for (uint32_t t = 0; t < rounds; t++) {
        const uint32_t out = in > p->row ? in / 2 : 1u << (log2_ceil(in) - 1);
        rs.in[t] = in;
        rs.out[t] = out;
        rs.chunk0[t] = chunks;
        chunks += (out + 63) / 64;
        if (p->weights == GRAPE_SHORT_FULL) {
            const bool rows = in > p->row;
            rs.rowlen[t] = rows ? p->row : 1;
            rs.rowpad[t] = rows ? 1u << row_log : 1;
        } else if (p->weights == GRAPE_SHORT_ROWS && in > p->row) {
            rs.rowlen[t] = p->row;
        }
        rs.off[t + 1] = (uint32_t)total;
        total += out;
        in = out;
    }
    rs.chunk0[rounds] = chunks;
    if (p->weights) GRAPE_REQUIRE(p->top_level + 1 >= (p->weights == GRAPE_SHORT_FULL ? rounds : rows_log) && p->top_level < 30, "the pyramid has no level for every round");
    hipStream_t s = as_stream(st);
    void* ws;
    int rc = scratch_get(kSlotShort, 32 * ((size_t)nt * total + (size_t)chunks * NV), &ws, s);
    if (rc) return rc;
    uint32_t* partial = (uint32_t*)ws + 8 * (size_t)nt * total;

    FoldSeg f = {};
    for (int k = 0; k < nt; k++) {
        f.src[k] = p->x[k];
        f.lev[k] = (uint32_t*)ws + 8 * (size_t)k * total;
        rs.x[k] = p->x[k];
        rs.lev[k] = f.lev[k];
    }
    f.v_end = p->v_end;
    for (uint32_t t = 1; t <= rounds; t++) f.off[t] = rs.off[t];
    for (uint32_t t = 0; t < rounds;) {
        // rows of a length that is no power of two are folded onto one row first: the padded row has another stride
        const bool rows = rs.in[t] > p->row && (p->row & (p->row - 1)) != 0;
        const uint32_t vars = rows ? rows_log - t : rounds - t;
        const uint32_t full = rows ? rs.in[t] : 1u << vars;
        f.live = rs.in[t];
        f.k = vars < kLevelVars ? vars : kLevelVars;
        f.stride = full >> f.k;
        f.t0 = t;
        const uint32_t need = log2_ceil(f.stride);
        f.cshift = kLevelVars - f.k < need ? kLevelVars - f.k : need;
        fold_levels_kernel<<<dim3((f.stride + (1u << f.cshift) - 1) >> f.cshift, nt), kBlock, 0, s>>>(f);
        t += f.k;
        for (int k = 0; k < nt; k++) f.src[k] = f.lev[k] + 8 * (size_t)f.off[t];
    }

    rs.beta = p->beta;
    rs.pyramid = p->pyramid;
    rs.partial = partial;
    rs.rounds = rounds;
    rs.top_level = p->top_level;
    RoundFinish fin = {};
    fin.partial = partial;
    fin.sums = p->sums;
    fin.stride = p->stride;
    fin.rounds = rounds;
    for (uint32_t t = 0; t <= rounds; t++) fin.chunk0[t] = rs.chunk0[t];
    bool any_last = false;
    for (int k = 0; k < nt; k++) {
        fin.end[k] = rs.lev[k] + 8 * (size_t)rs.off[rounds];
        fin.last[k] = p->last[k];
        fin.copy[k] = p->last_copy[k];
        any_last |= fin.last[k] || fin.copy[k];
    }
    const unsigned nfin = rounds + (any_last ? 1 : 0);
    if (table) {
        round_sums_kernel<true, true><<<chunks, 384, 0, s>>>(rs);
        round_finish_kernel<8><<<nfin, kBlock, 0, s>>>(fin);
    } else if (logup) {
        round_sums_kernel<true, false><<<chunks, 192, 0, s>>>(rs);
        round_finish_kernel<5><<<nfin, kBlock, 0, s>>>(fin);
    } else {
        round_sums_kernel<false, false><<<chunks, 192, 0, s>>>(rs);
        round_finish_kernel<3><<<nfin, kBlock, 0, s>>>(fin);
    }
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
