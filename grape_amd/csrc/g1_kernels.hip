// G1 kernels: generator derivation, fixed-base tables and the Hyrax row-commitment kernels.
//
// Commitment design (one GPU, 288 GB of HBM): all rows of a matrix are committed against the
// SAME generators, so the work per scalar is bought down with memory — a table of
// k * 2^(c*w) * G_i for every digit value k and window w turns each signed radix-2^c digit into
// exactly one mixed addition into a single per-lane accumulator (no per-window accumulators,
// no doubling chain at the end).  For int16-range weights c = 16 makes that one addition per
// matrix element.  Lanes own columns (coalesced scalar reads), accumulate in extended Jacobian
// (XYZZ) coordinates, and a second kernel folds the 64 lane partials of each row and maps the
// result to affine coordinates.
#define GRAPE_FP_MUL_OUTLINE 1
#include "common.hpp"
#include "commit_geometry.hpp"
#include "fp30.hpp"
#include "fr26.hpp"
#include "quad30.hpp"

namespace grape {

// The one shared body of the Fp multiplier / squarer (about a thousand instructions each, so
// every branch inside stays short-range).
__device__ __noinline__ Fp fp_mul_outline(Fp a, Fp b) { return mul(a, b); }
__device__ __noinline__ Fp fp_sqr_outline(Fp a) { return sqr(a); }

// Memory images in 32-bit words: an Fp element is FW words (12 for BLS12-381, 8 for BN254), an
// affine point 2 FW, a Jacobian point 3 FW, an XYZZ point 4 FW; L30 is the limb count of the
// working form of fp30.hpp.
constexpr int FW = FpParams::N;
constexpr int L30 = fp30::N;

__device__ __forceinline__ Fp ld_fp(const uint32_t* p) {
    const uint4* q = reinterpret_cast<const uint4*>(p);
    Fp r;
#pragma unroll
    for (int i = 0; i < FW / 4; i++) {
        const uint4 a = q[i];
        r.v[4 * i] = a.x; r.v[4 * i + 1] = a.y; r.v[4 * i + 2] = a.z; r.v[4 * i + 3] = a.w;
    }
    return r;
}
__device__ __forceinline__ void st_fp(uint32_t* p, const Fp& a) {
    uint4* q = reinterpret_cast<uint4*>(p);
#pragma unroll
    for (int i = 0; i < FW / 4; i++) q[i] = make_uint4(a.v[4 * i], a.v[4 * i + 1], a.v[4 * i + 2], a.v[4 * i + 3]);
}
__device__ __forceinline__ G1Affine ld_affine(const uint32_t* base, size_t i) {
    G1Affine r;
    r.x = ld_fp(base + 2 * FW * i);
    r.y = ld_fp(base + 2 * FW * i + FW);
    return r;
}
__device__ __forceinline__ void st_affine(uint32_t* base, size_t i, const G1Affine& p) {
    st_fp(base + 2 * FW * i, p.x);
    st_fp(base + 2 * FW * i + FW, p.y);
}
__device__ __forceinline__ G1Xyzz ld_xyzz(const uint32_t* base, size_t i) {
    G1Xyzz r;
    r.x = ld_fp(base + 4 * FW * i);
    r.y = ld_fp(base + 4 * FW * i + FW);
    r.zz = ld_fp(base + 4 * FW * i + 2 * FW);
    r.zzz = ld_fp(base + 4 * FW * i + 3 * FW);
    return r;
}
__device__ __forceinline__ void st_xyzz(uint32_t* base, size_t i, const G1Xyzz& p) {
    st_fp(base + 4 * FW * i, p.x);
    st_fp(base + 4 * FW * i + FW, p.y);
    st_fp(base + 4 * FW * i + 2 * FW, p.zz);
    st_fp(base + 4 * FW * i + 3 * FW, p.zzz);
}
__device__ __forceinline__ Fr ld_fr8(const uint32_t* base, size_t i) {
    const uint4* p = reinterpret_cast<const uint4*>(base) + 2 * i;
    uint4 lo = p[0], hi = p[1];
    Fr r;
    r.v[0] = lo.x; r.v[1] = lo.y; r.v[2] = lo.z; r.v[3] = lo.w;
    r.v[4] = hi.x; r.v[5] = hi.y; r.v[6] = hi.z; r.v[7] = hi.w;
    return r;
}

// Wide-table entry: an affine point in the working form, x[L30] then y[L30] as 32-bit
// words.  BLS12-381's 104 bytes are padded to 128, so that every gather is exactly one cache line;
// BN254's 72 bytes are stored in 80 (a multiple of 16 bytes: the loads stay aligned, half of the
// entries straddle two lines) - the table is 37.5 % smaller, which is what lets 15-bit windows fit
// the table budget there.
constexpr int kWideEntryWords = (2 * L30 <= 20) ? 20 : 32;
static_assert(kWideEntryWords % 4 == 0 && kWideEntryWords >= 2 * L30, "entry layout");
__device__ __forceinline__ Affine30 ld_entry30(const uint32_t* table, size_t e) {
    const uint4* q = reinterpret_cast<const uint4*>(table + (size_t)kWideEntryWords * e);
    uint4 w[(2 * L30 + 3) / 4];
#pragma unroll
    for (int i = 0; i < (2 * L30 + 3) / 4; i++) w[i] = q[i];
    const uint32_t* f = reinterpret_cast<const uint32_t*>(w);
    Affine30 r;
#pragma unroll
    for (int i = 0; i < L30; i++) {
        r.x.v[i] = (int32_t)f[i];
        r.y.v[i] = (int32_t)f[L30 + i];
    }
    return r;
}
// coordinates in [0, p), balanced
__device__ __forceinline__ void st_entry30_raw(uint32_t* table, size_t e, const Affine30& a) {
    uint32_t f[kWideEntryWords];
#pragma unroll
    for (int i = 0; i < L30; i++) {
        f[i] = (uint32_t)a.x.v[i];
        f[L30 + i] = (uint32_t)a.y.v[i];
    }
#pragma unroll
    for (int i = 2 * L30; i < kWideEntryWords; i++) f[i] = 0;
    uint4* q = reinterpret_cast<uint4*>(table + (size_t)kWideEntryWords * e);
#pragma unroll
    for (int i = 0; i < kWideEntryWords / 4; i++) q[i] = make_uint4(f[4 * i], f[4 * i + 1], f[4 * i + 2], f[4 * i + 3]);
}
__device__ __forceinline__ void st_entry30(uint32_t* table, size_t e, const G1Affine& a) {
    st_entry30_raw(table, e, Affine30{fp30::from_canonical(a.x), fp30::from_canonical(a.y)});
}
__device__ __forceinline__ bool entry_is_inf(const Affine30& a) {
    uint32_t z = 0;
#pragma unroll
    for (int i = 0; i < L30; i++) z |= (uint32_t)a.x.v[i] | (uint32_t)a.y.v[i];
    return z == 0;
}
// Per-lane partial accumulator in memory: x, y, zz, zzz (kCoordWords words each, a multiple of 8 bytes), the identity
// flag and padding = 64 words (256 bytes).
using geom::kPartialWords;
constexpr int kCoordWords = (L30 + 1) & ~1;
static_assert(4 * kCoordWords + 1 <= kPartialWords && kCoordWords % 2 == 0, "accumulator layout");
__device__ __forceinline__ void st_partial30(uint32_t* base, size_t i, const Xyzz30& a) {
    uint32_t f[kPartialWords];
#pragma unroll
    for (int k = 0; k < kPartialWords; k++) f[k] = 0;
#pragma unroll
    for (int k = 0; k < L30; k++) {
        f[k] = (uint32_t)a.x.v[k];
        f[kCoordWords + k] = (uint32_t)a.y.v[k];
        f[2 * kCoordWords + k] = (uint32_t)a.zz.v[k];
        f[3 * kCoordWords + k] = (uint32_t)a.zzz.v[k];
    }
    f[4 * kCoordWords] = a.inf ? 1u : 0u;
    uint4* q = reinterpret_cast<uint4*>(base + geom::partial_word(i));
#pragma unroll
    for (int k = 0; k < kPartialWords / 4; k++) q[k] = make_uint4(f[4 * k], f[4 * k + 1], f[4 * k + 2], f[4 * k + 3]);
}
__device__ __forceinline__ Xyzz30 ld_partial30(const uint32_t* base, size_t i) {
    const uint4* q = reinterpret_cast<const uint4*>(base + geom::partial_word(i));
    uint4 w[kCoordWords + 1];
#pragma unroll
    for (int k = 0; k < kCoordWords + 1; k++) w[k] = q[k];
    const uint32_t* f = reinterpret_cast<const uint32_t*>(w);
    Xyzz30 a;
#pragma unroll
    for (int k = 0; k < L30; k++) {
        a.x.v[k] = (int32_t)f[k];
        a.y.v[k] = (int32_t)f[kCoordWords + k];
        a.zz.v[k] = (int32_t)f[2 * kCoordWords + k];
        a.zzz.v[k] = (int32_t)f[3 * kCoordWords + k];
    }
    a.inf = f[4 * kCoordWords] != 0;
    return a;
}
// acc += q for two accumulators in the working form, exceptional cases through the canonical-form addition
__device__ __forceinline__ void padd30(Xyzz30& acc, const Xyzz30& q) {
    if (!xyzz30_add(acc, q)) {
        G1Xyzz c = xyzz30_to_canonical(acc);
        xyzz_add(c, xyzz30_to_canonical(q));
        acc = xyzz30_from_canonical(c);
    }
}

// acc += +-entry through the mixed addition of the working form; the rare exceptional step (entry = +-acc)
// goes through the exact canonical-form addition.
__device__ __forceinline__ void madd30(Xyzz30& acc, const Affine30& e, bool negate) {
    if (entry_is_inf(e)) return;
    if (!xyzz30_madd(acc, e, negate)) {
        G1Xyzz c = xyzz30_to_canonical(acc);
        G1Affine a;
        a.x = fp30::to_canonical(e.x);
        a.y = fp30::to_canonical(e.y);
        xyzz_add_affine(c, a, negate);
        acc = xyzz30_from_canonical(c);
    }
}

// acc += k * G_col for a canonical (non-Montgomery) 255-bit scalar k: signed radix-2^c digits,
// one gather and one mixed addition per non-zero digit.
// One signed radix-2^c digit of a canonical scalar: window w, incoming carry -> magnitude, sign,
// outgoing carry.
__device__ __forceinline__ uint32_t fr_digit(const Fr& k, uint32_t w, uint32_t c, uint32_t& carry, bool& neg) {
    const uint32_t half = 1u << (c - 1), mask = (1u << c) - 1u;
    const uint32_t bit = w * c;
    // c <= 16 bits starting at `bit`, possibly straddling two limbs
    const uint32_t limb = bit >> 5, sh = bit & 31;
    uint32_t lo = 0, hi = 0;
#pragma unroll
    for (int q = 0; q < 8; q++) {
        lo = (q == (int)limb) ? k.v[q] : lo;
        hi = (q == (int)limb + 1) ? k.v[q] : hi;
    }
    const uint64_t both = ((uint64_t)hi << 32) | lo;
    const uint32_t d = ((uint32_t)(both >> sh) & mask) + carry;
    neg = d > half;                      // digit in (half, 2^c] -> d - 2^c, carry 1
    carry = neg ? 1u : 0u;
    return neg ? (mask + 1u - d) : d;
}

// acc += k * G_col through the wide table: one gather and one mixed addition per non-zero digit.
// While the addition of digit w runs, the table line of digit w+1 is already on its way (one
// word of it is touched right after the entry of digit w has been requested).  Only the digits w0 .. w1 - 1 are added.
__device__ __forceinline__ void madd_scalar_fr(Xyzz30& acc, const Fr& k_in, const uint32_t* table, size_t N, uint32_t col,
                                               uint32_t c, uint32_t nw, uint32_t K, int* err_flag, uint32_t w0 = 0, uint32_t w1 = ~0u) {
    // The scalar is taken as +-|k| with |k| <= (r-1)/2 < 2^254 (r - k and the negated point when k is
    // in the upper half): the top window then never carries out, and nw = ceil(255/c) windows are
    // enough - one addition fewer per scalar at c = 15.
    Fr k = k_in;
    uint32_t borrow = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t half_i = (FrParams::mod(i) >> 1) | (i + 1 < 8 ? FrParams::mod(i + 1) << 31 : 0u);
        const uint64_t t = (uint64_t)half_i - (uint64_t)k.v[i] - (uint64_t)borrow;
        borrow = (uint32_t)(t >> 63);
    }
    const bool flip = borrow != 0;                        // k > (r-1)/2
    k = cneg(k, flip);
    uint32_t nwin = nw;
    while (nwin > 0 && (nwin - 1) * c >= 256) nwin--;     // windows that start inside the scalar
    const uint32_t end = w1 < nwin ? w1 : nwin;
    uint32_t carry = 0;
    bool neg = false;
    for (uint32_t w = 0; w < w0 && w < end; w++) (void)fr_digit(k, w, c, carry, neg);
    neg = false;
    uint32_t mag = w0 < end ? fr_digit(k, w0, c, carry, neg) : 0;
    uint32_t touch = 0;
    for (uint32_t w = w0; w < end; w++) {
        bool neg_n = false;
        const uint32_t mag_n = (w + 1 < end) ? fr_digit(k, w + 1, c, carry, neg_n) : 0;
        if (mag != 0) {
            if (mag > K) {
                *err_flag = 1;
            } else {
                const Affine30 e = ld_entry30(table, geom::table_entry(w, K, mag, N, col));
                // unconditional, so that the compiler counts the outstanding loads exactly
                const size_t nxt = (mag_n != 0 && mag_n <= K) ? geom::table_entry(w + 1, K, mag_n, N, col) : (size_t)col;
                touch = table[(size_t)kWideEntryWords * nxt];
                if (kWideEntryWords % 32 != 0) touch |= table[(size_t)kWideEntryWords * nxt + kWideEntryWords - 1];   // dense entries: both lines
                madd30(acc, e, neg != flip);
            }
        }
        mag = mag_n;
        neg = neg_n;
    }
    asm volatile("" ::"v"(touch));      // keeps the last touch alive until here
    if (carry && end == nwin) *err_flag = 1;   // cannot happen for canonical scalars when nw*c >= 255
}

__device__ __forceinline__ G1Xyzz shfl_down_xyzz(const G1Xyzz& a, int off) {
    G1Xyzz r;
#pragma unroll
    for (int i = 0; i < FW; i++) {
        r.x.v[i] = __shfl_down(a.x.v[i], off, 64);
        r.y.v[i] = __shfl_down(a.y.v[i], off, 64);
        r.zz.v[i] = __shfl_down(a.zz.v[i], off, 64);
        r.zzz.v[i] = __shfl_down(a.zzz.v[i], off, 64);
    }
    return r;
}

// The group operations are always inlined into the kernels; only the Fp multiplier and squarer
// are out-of-line.  An out-of-line device function large enough to need far branches is not
// safe: the compiler's far-branch expansion inside a non-kernel function borrows s[30:31] - the
// return address - so such a function never returns once the far path is taken (seen in the
// generated code of an out-of-line mixed addition: the "accumulator is at infinity for every
// active lane" path jumped through s[30:31] and the final s_setpc_b64 s[30:31] then looped
// forever).  Kernels have no return address to lose, and the multiplier body is far below the
// +-128 KiB range of a short branch.
__device__ __forceinline__ void madd(G1Xyzz& acc, const G1Affine& p, bool negate) { xyzz_add_affine(acc, p, negate); }
__device__ __forceinline__ void padd(G1Xyzz& acc, const G1Xyzz& q) { xyzz_add(acc, q); }
__device__ __forceinline__ void pdbl(G1Xyzz& acc) { xyzz_dbl(acc); }
// 1/a for a canonical, non-zero a: through the working form and its divstep inversion (about ten
// thousand instructions) instead of the a^(p-2) ladder on saturated limbs (about six hundred thousand)
__device__ __forceinline__ Fp fp_inverse_fast(const Fp& a) {
    return fp30::to_canonical(fp30::inverse_by(fp30::from_canonical_lazy(a)));
}
__device__ __forceinline__ G1Affine to_affine(const G1Xyzz& p) {
    if (p.is_inf()) return G1Affine::inf();
    return xyzz_to_affine_with_inv(p, fp_inverse_fast(p.zzz));
}

// k * P for a 256-bit canonical scalar held in 8 limbs
__device__ __forceinline__ G1Xyzz scalar_mul(const G1Affine& p, const uint32_t* k, int top_bit) {
    G1Xyzz acc = G1Xyzz::inf();
    for (int i = top_bit; i >= 0; i--) {
        pdbl(acc);
        if ((k[i >> 5] >> (i & 31)) & 1) madd(acc, p, false);
    }
    return acc;
}

__global__ void __launch_bounds__(64) scalar_mul_base_kernel(uint32_t* out, const uint32_t* k, const uint32_t* base, size_t n) {
    size_t i = (size_t)blockIdx.x * 64 + threadIdx.x;
    if (i >= n) return;
    uint32_t kk[8];
#pragma unroll
    for (int j = 0; j < 8; j++) kk[j] = k[8 * i + j];
    G1Affine p = ld_affine(base, 0);
    st_affine(out, i, to_affine(scalar_mul(p, kk, 255)));
}

// bases[w*N + i] = 2^(c*w) * G_i, affine
__global__ void __launch_bounds__(64) window_bases_kernel(uint32_t* bases, const uint32_t* gens, size_t N, uint32_t c, uint32_t nw) {
    size_t i = (size_t)blockIdx.x * 64 + threadIdx.x;
    if (i >= N) return;
    G1Affine g = ld_affine(gens, i);
    st_affine(bases, i, g);
    G1Xyzz cur = G1Xyzz::from_affine(g);
    for (uint32_t w = 1; w < nw; w++) {
        for (uint32_t d = 0; d < c; d++) pdbl(cur);
        st_affine(bases, (size_t)w * N + i, to_affine(cur));
    }
}

// One thread per (window w, generator i, chunk j): XYZZ multiples k*B for k = j*CH+1 .. j*CH+CH
// (clipped to K) into tmp[((j - j0)*CH + t) * (nw*N) + w*N + i].
__global__ void __launch_bounds__(64) wide_chain_kernel(uint32_t* tmp, const uint32_t* bases, size_t N, uint32_t nw, uint32_t K,
                                                        uint32_t CH, uint32_t j0, uint32_t nj) {
    size_t tid = (size_t)blockIdx.x * 64 + threadIdx.x;
    size_t per_chunk = (size_t)nw * N;
    if (tid >= per_chunk * nj) return;
    uint32_t jj = (uint32_t)(tid / per_chunk);
    size_t wi = tid - (size_t)jj * per_chunk;       // w*N + i
    uint32_t j = j0 + jj;
    G1Affine B = ld_affine(bases, wi);
    uint32_t kstart[8] = {j * CH + 1, 0, 0, 0, 0, 0, 0, 0};
    G1Xyzz acc = scalar_mul(B, kstart, 31 - __clz((int)kstart[0]));
    for (uint32_t t = 0; t < CH; t++) {
        uint32_t k = j * CH + 1 + t;
        if (k > K) break;
        st_xyzz(tmp, ((size_t)jj * CH + t) * per_chunk + wi, acc);
        madd(acc, B, false);
    }
}

// Batched XYZZ -> affine (Montgomery's trick over 8 entries per thread, strided so that lanes
// stay adjacent).  Entry e of tmp goes to dst[map(e)] where, for the wide table,
// e = (jj*CH + t)*(nw*N) + w*N + i  ->  ((w*K) + (j0*CH + jj*CH + t))*N + i.
constexpr int kNormChunk = 8;
__global__ void __launch_bounds__(64) wide_normalize_kernel(uint32_t* table, const uint32_t* tmp, size_t N, uint32_t nw, uint32_t K,
                                                            uint32_t CH, uint32_t j0, size_t n_entries) {
    size_t t0 = (size_t)blockIdx.x * 64 + threadIdx.x;
    size_t nthreads = (n_entries + kNormChunk - 1) / kNormChunk;
    if (t0 >= nthreads) return;
    Fp pre[kNormChunk];
    Fp acc = Fp::one();
#pragma unroll
    for (int k = 0; k < kNormChunk; k++) {
        size_t e = t0 + (size_t)k * nthreads;
        pre[k] = acc;
        if (e < n_entries) {
            Fp zzz = ld_fp(tmp + 4 * FW * e + 3 * FW);
            if (!zzz.is_zero()) acc = fmul(acc, zzz);
        }
    }
    Fp inv = fp_inverse_fast(acc);
    const size_t per_chunk = (size_t)nw * N;
#pragma unroll
    for (int k = kNormChunk - 1; k >= 0; k--) {
        size_t e = t0 + (size_t)k * nthreads;
        if (e >= n_entries) continue;
        G1Xyzz p = ld_xyzz(tmp, e);
        size_t kk = e / per_chunk;                  // jj*CH + t
        size_t wi = e - kk * per_chunk;
        size_t w = wi / N, i = wi - w * N;
        size_t kidx = (size_t)j0 * CH + kk;         // k - 1
        if (kidx >= K) continue;
        G1Affine a = G1Affine::inf();
        if (!p.zzz.is_zero()) {
            Fp zi = fmul(inv, pre[k]);
            inv = fmul(inv, p.zzz);
            a = xyzz_to_affine_with_inv(p, zi);
        }
        st_entry30(table, (w * K + kidx) * N + i, a);
    }
}

// ------------------------------------------------------------------------------------------------
// Table generation by levels: once the multiples 1..have of every base are in the table, the next
// cnt <= have are E[have + k] = E[k] + E[have] (k = have is the doubling of E[have]) - additions
// of two AFFINE entries that are already final, all independent.  An affine addition is 3M + 1S
// once the inverse of its slope's denominator is known, and Montgomery's trick shares one
// inversion over a thread's run of consecutive k: a forward pass multiplies the denominators up,
// parking every prefix product in the destination entry it belongs to (free until the backward
// pass fills it), one divstep inversion, and a backward pass that peels the inverses off and
// writes the sums.  About 6 products and 0.5 KB of traffic per entry, where a chain of mixed
// XYZZ additions plus the normalisation of every entry costs 17 products and an inversion per 8.
// A run whose denominators multiply to zero (a base that is the identity or has small order: no
// generator of the prime-order group) raises *degenerate and leaves its entries to
// wide_extend_exact_kernel.
// ------------------------------------------------------------------------------------------------
constexpr uint32_t kExtendRun = 64;   // additions that share one inversion
constexpr uint32_t kFirstChain = 16;  // multiples of a base made by the chain of mixed additions before the levels start
constexpr int kFp30Quads = (L30 + 3) / 4;
__device__ __forceinline__ Fp30 ld_fp30(const uint32_t* p) {
    const uint4* q = reinterpret_cast<const uint4*>(p);
    uint4 w[kFp30Quads];
#pragma unroll
    for (int i = 0; i < kFp30Quads; i++) w[i] = q[i];
    const uint32_t* f = reinterpret_cast<const uint32_t*>(w);
    Fp30 r;
#pragma unroll
    for (int i = 0; i < L30; i++) r.v[i] = (int32_t)f[i];
    return r;
}
__device__ __forceinline__ void st_fp30(uint32_t* p, const Fp30& a) {
    uint32_t f[4 * kFp30Quads];
#pragma unroll
    for (int i = 0; i < 4 * kFp30Quads; i++) f[i] = i < L30 ? (uint32_t)a.v[i] : 0u;
    uint4* q = reinterpret_cast<uint4*>(p);
#pragma unroll
    for (int i = 0; i < kFp30Quads; i++) q[i] = make_uint4(f[4 * i], f[4 * i + 1], f[4 * i + 2], f[4 * i + 3]);
}
static_assert(4 * kFp30Quads <= kWideEntryWords, "a prefix product must fit the entry it is parked in");

// One thread per (run of `run` consecutive k, window w, generator i); i is the fastest index, so a
// wave reads and writes adjacent entries.
__global__ void __launch_bounds__(kBlock, 2) wide_extend_kernel(uint32_t* table, size_t N, uint32_t nw, uint32_t K, uint32_t have,
                                                             uint32_t cnt, uint32_t run, int* degenerate) {
    const size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x;
    const size_t per = (size_t)nw * N;
    const uint32_t nruns = (cnt + run - 1) / run;
    if (t >= per * nruns) return;
    const uint32_t r = (uint32_t)(t / per);
    const size_t wi = t - (size_t)r * per;
    const size_t w = wi / N, i = wi - w * N;
    const uint32_t k0 = r * run + 1;                              // first k of the run
    const uint32_t k1 = k0 + run < cnt + 1 ? k0 + run : cnt + 1;  // one past its last
    const size_t e0 = w * K * N + i;                              // entry of the multiple k: e0 + (k-1) N
    const Affine30 f = ld_entry30(table, e0 + (size_t)(have - 1) * N);
    bool bad = entry_is_inf(f);
    Fp30 acc = fp30::one();
    for (uint32_t k = k0; k < k1; k++) {
        const Affine30 e = ld_entry30(table, e0 + (size_t)(k - 1) * N);
        bad |= entry_is_inf(e);
        st_fp30(table + (size_t)kWideEntryWords * (e0 + (size_t)(have + k - 1) * N), acc);
        acc = fp30::mul(acc, affine30_slope_den(e, f, k == have));
    }
    bad |= fp30::is_zero_mod_p(acc);
    if (bad) {
        *degenerate = 1;
        return;
    }
    Fp30 inv = fp30::inverse_by(acc);
    for (uint32_t k = k1 - 1; k >= k0; k--) {
        const size_t dst = e0 + (size_t)(have + k - 1) * N;
        const Affine30 e = ld_entry30(table, e0 + (size_t)(k - 1) * N);
        const Fp30 dinv = fp30::mul(inv, ld_fp30(table + (size_t)kWideEntryWords * dst));
        inv = fp30::mul(inv, affine30_slope_den(e, f, k == have));
        const Affine30 sum = affine30_add_given_inverse(e, f, k == have, dinv);
        st_entry30_raw(table, dst, Affine30{fp30::balance(sum.x), fp30::balance(sum.y)});
    }
}

// The same level through the general addition, one thread per entry, every exceptional case
// handled (identity, equal and opposite points): runs only when the level met a degenerate run.
__global__ void __launch_bounds__(64) wide_extend_exact_kernel(uint32_t* table, size_t N, uint32_t nw, uint32_t K, uint32_t have,
                                                               uint32_t cnt, const int* degenerate) {
    if (*degenerate == 0) return;
    const size_t per = (size_t)nw * N;
    for (size_t t = (size_t)blockIdx.x * 64 + threadIdx.x; t < per * cnt; t += (size_t)gridDim.x * 64) {
        const uint32_t k = (uint32_t)(t / per) + 1;
        const size_t wi = t - (size_t)(k - 1) * per;
        const size_t w = wi / N, i = wi - w * N;
        const size_t e0 = w * K * N + i;
        Xyzz30 acc = xyzz30_inf();
        madd30(acc, ld_entry30(table, e0 + (size_t)(k - 1) * N), false);
        madd30(acc, ld_entry30(table, e0 + (size_t)(have - 1) * N), false);
        st_entry30(table, e0 + (size_t)(have + k - 1) * N, xyzz30_to_affine(acc));
    }
}

// Reference-format table from a one-window wide table over the generators i0 .. i0+ns:
// out[w*N + i0 + i] = w * G_(i0+i) in the canonical memory form (w = 0: the identity), one product
// per coordinate to change the limb form and the Montgomery radix.
__global__ void __launch_bounds__(kBlock) ref_from_wide_kernel(uint32_t* out, const uint32_t* wide, size_t N, size_t i0, size_t ns, uint32_t W) {
    const size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (t >= ns * W) return;
    const size_t w = t / ns, i = t - w * ns;
    G1Affine a = G1Affine::inf();
    if (w > 0) {
        const Affine30 e = ld_entry30(wide, (w - 1) * ns + i);
        a.x = fp30::to_canonical(e.x);
        a.y = fp30::to_canonical(e.y);
    }
    st_affine(out, w * N + i0 + i, a);
}

// ------------------------------------------------------------------------------------------------
// commitment, wide table
// ------------------------------------------------------------------------------------------------
// Each wave owns one row segment of `seg` columns; lane l takes columns l, l+64, ...
// partial[(row*nseg + s)*64 + lane] receives the lane's XYZZ accumulator; full-width scalars of few rows go over split.parts
// waves per segment (geom::window_split), partial[((row*nseg + s)*parts + part)*64 + lane].
// BASED (digits that are table indices): elements of index base1 cost nothing, the rows' sums are added to `start` instead (see
// grape_commit_indexed), on their way to affine coordinates: a lane that began with it would make a full addition of its first
// entry where the others take theirs over, 1.5 % of a row of 4096 and twice the time of one of 256.  Where the rows are uneven the workgroups are one wave, dealt by geom::spread_unit: a row that is all
// padding is over at once, and beside three full ones in a workgroup, or on the same engine every time, its place would stay
// empty.  2048 rows of 11008 padded to 16384, a third of 2^25 elements the padding's: a range lookup 6.28 -> 5.40 ms.  (Even
// rows keep the order of the launch: a mapping lookup of 2^27 takes 25.3 ms that way and 25.8 dealt.)
struct CommitBase {
    const uint32_t* start;      // an accumulator
    int32_t base1;
    size_t step;                // of the deal, or 0
};
template <bool FR, bool BASED = false>
__global__ void __launch_bounds__(kBlock) commit_wide_kernel(uint32_t* partial, const void* scalars, uint32_t rowlen, size_t rows,
                                                             uint32_t seg, uint32_t nseg, const uint32_t* table, size_t N,
                                                             uint32_t c, uint32_t nw, uint32_t K, int* err_flag, geom::WindowSplit split, CommitBase base) {
    const int lane = threadIdx.x & 63;
    const size_t wave = BASED && base.step ? geom::spread_unit(blockIdx.x, gridDim.x, base.step) : ((size_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
    const uint32_t parts = FR ? split.parts : 1;
    if (wave >= rows * nseg * parts) return;
    const size_t unit = FR ? wave / parts : wave;
    const uint32_t w0 = (uint32_t)(wave - unit * parts) * split.per;
    const geom::WaveSpan span = geom::wave_span(unit, nseg, seg, rowlen);
    const size_t row = span.row;
    const uint32_t s = span.s, col_end = span.col_end;
    const uint32_t half = 1u << (c - 1), mask = (c == 32) ? 0xffffffffu : ((1u << c) - 1u);
    Xyzz30 acc = xyzz30_inf();
    auto digits_of = [&](uint32_t col) { return ((const int32_t*)scalars)[geom::scalar_index(row, rowlen, col)]; };
    // where a digit is used, not where it is loaded: there it would wait for the load
    auto without_base = [&](int32_t x) { return BASED && x == base.base1 ? 0 : x; };
    // int path: the scalars of the next two columns are kept in flight (the next one addresses
    // the table line to touch, the one after is being loaded)
    int32_t sc1 = 0, sc2 = 0;
    if (!FR) {
        const uint32_t c0 = s * seg + lane;
        if (c0 + 64 < col_end) sc1 = digits_of(c0 + 64);
        if (c0 + 128 < col_end) sc2 = digits_of(c0 + 128);
    }
    int32_t sc0 = (!FR && s * seg + lane < col_end) ? digits_of(s * seg + lane) : 0;
    // destination of the look-ahead touches: one register for the whole loop, read only after it.  (Declared
    // inside the loop it is free again at the top of the next iteration, the compiler reuses it for an
    // address there and has to wait for every outstanding load first - 1.5 % of the kernel's time.)
    uint32_t touch = 0;
    for (uint32_t col = s * seg + lane; col < col_end; col += 64) {
        if (FR) {
            const Fr k = from_mont(ld_fr8((const uint32_t*)scalars, geom::scalar_index(row, rowlen, col)));
            madd_scalar_fr(acc, k, table, N, col, c, nw, K, err_flag, w0, w0 + split.per);
        } else {
            int64_t v = without_base(sc0);
            const int64_t v_next = without_base(sc1);
            sc0 = sc1;
            sc1 = sc2;
            sc2 = (col + 192 < col_end) ? digits_of(col + 192) : 0;
            // The table line of the NEXT column's first digit is touched (one word) right after
            // this column's own entry is requested, so that it is in cache when its turn comes:
            // with two waves per SIMD an exposed HBM round trip per addition costs issue slots.
            // (the touch is unconditional - a column without a successor touches its own first
            // table line - because the compiler counts outstanding loads exactly only in
            // straight-line code; a conditional load after the entry's would make it wait for both)
            size_t next_entry = col;
            bool have_next = false;
            if (col + 64 < col_end) {
                int64_t vn = v_next;
                int64_t dn = vn & (int64_t)mask;
                vn >>= c;
                if (dn > (int64_t)half || (dn == (int64_t)half && vn < 0)) dn -= (int64_t)mask + 1;
                const uint32_t magn = (uint32_t)(dn < 0 ? -dn : dn);
                have_next = magn != 0 && magn <= K;
                if (have_next) next_entry = geom::table_entry(0, K, magn, N, col + 64);
            }
            const uint32_t* touch_ptr = table + (size_t)kWideEntryWords * next_entry;
            for (uint32_t w = 0; w < nw; w++) {
                int64_t d = v & (int64_t)mask;
                v >>= c;                            // arithmetic shift keeps the sign
                // digits above half go negative with a carry; exactly half goes negative only
                // when what remains is negative (so that -2^(c-1) recodes to one digit)
                if (d > (int64_t)half || (d == (int64_t)half && v < 0)) {
                    d -= (int64_t)mask + 1;
                    v += 1;
                }
                const bool neg = d < 0;
                const uint32_t mag = (uint32_t)(neg ? -d : d);
                if (mag != 0) {
                    if (mag > K) { *err_flag = 1; continue; }
                    const Affine30 e = ld_entry30(table, geom::table_entry(w, K, mag, N, col));
                    touch = *touch_ptr;
                    if (kWideEntryWords % 32 != 0) touch |= touch_ptr[kWideEntryWords - 1];   // dense entries: both lines
                    madd30(acc, e, neg);
                }
            }
            if (v != 0) *err_flag = 1;              // scalar does not fit nw windows
        }
    }
    asm volatile("" ::"v"(touch));                  // keeps the touches alive until here
    st_partial30(partial, wave * 64 + lane, acc);
}

__global__ void commit_start_kernel(uint32_t* out, const uint32_t* affine) {
    const G1Affine a = ld_affine(affine, 0);
    st_partial30(out, 0, a.is_inf() ? xyzz30_inf() : xyzz30_from_canonical(G1Xyzz{a.x, a.y, Fp::one(), Fp::one()}));
}

// Scaled table: out[t*ncols + i] = s_t * G_i for a short list of scalars s_t (Montgomery Fr).
// Stage 1 leaves XYZZ points (canonical form) in tmp[(t - t0)*ncols + i]; stage 2 normalises
// 8 per thread and writes 128-byte working-form entries.
__global__ void __launch_bounds__(kBlock) scaled_chain_kernel(uint32_t* tmp, const uint32_t* scalars, size_t t0, size_t nt,
                                                              size_t ncols, const uint32_t* table, size_t N, uint32_t c,
                                                              uint32_t nw, uint32_t K, int* err_flag) {
    size_t tid = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (tid >= nt * ncols) return;
    const size_t tt = tid / ncols;
    const uint32_t col = (uint32_t)(tid - tt * ncols);
    const Fr k = from_mont(ld_fr8(scalars, t0 + tt));
    Xyzz30 acc = xyzz30_inf();
    madd_scalar_fr(acc, k, table, N, col, c, nw, K, err_flag);
    st_xyzz(tmp, tid, xyzz30_to_canonical(acc));
}
__global__ void __launch_bounds__(64) scaled_normalize_kernel(uint32_t* out, const uint32_t* tmp, size_t e0, size_t n_entries) {
    size_t t0 = (size_t)blockIdx.x * 64 + threadIdx.x;
    size_t nthreads = (n_entries + kNormChunk - 1) / kNormChunk;
    if (t0 >= nthreads) return;
    Fp pre[kNormChunk];
    Fp acc = Fp::one();
#pragma unroll
    for (int k = 0; k < kNormChunk; k++) {
        size_t e = t0 + (size_t)k * nthreads;
        pre[k] = acc;
        if (e < n_entries) {
            Fp zzz = ld_fp(tmp + 4 * FW * e + 3 * FW);
            if (!zzz.is_zero()) acc = fmul(acc, zzz);
        }
    }
    Fp inv = fp_inverse_fast(acc);
#pragma unroll
    for (int k = kNormChunk - 1; k >= 0; k--) {
        size_t e = t0 + (size_t)k * nthreads;
        if (e >= n_entries) continue;
        G1Xyzz p = ld_xyzz(tmp, e);
        G1Affine a = G1Affine::inf();
        if (!p.zzz.is_zero()) {
            Fp zi = fmul(inv, pre[k]);
            inv = fmul(inv, p.zzz);
            a = xyzz_to_affine_with_inv(p, zi);
        }
        st_entry30(out, e0 + e, a);
    }
}

// ------------------------------------------------------------------------------------------------
// commitment, strided table (full-width scalars)
// ------------------------------------------------------------------------------------------------
// A per-window table spends its bytes on ceil(255/c) sets of 2^(c-1) multiples.  Keeping only every
// J-th set - entries k * 2^(c J q) * G_i for q < nsets = ceil(nw / J) - leaves room for wider windows
// within the same bytes: window w = q J + j is looked up in set q, and the J residues j get their own
// sums A_j, combined per row as sum_j 2^(c j) A_j by a Horner chain of (J - 1) c doublings.  With
// 4096 generators c = 16, J = 4 is 16 additions per scalar from 68 GB where the per-window table
// gives 19 from 82 GB; with 262144 generators c = 12, J = 22 (one set, 68 GB) is 22 additions where
// no per-window table above c = 8 fits.
//
// Digits are taken carry-free: with H = sum_w 2^(c w + c - 1), digit_w = ((k + H) >> c w mod 2^c) - 2^(c-1)
// lies in [-2^(c-1), 2^(c-1)) and sum_w digit_w 2^(c w) = k, so any window can be read on its own.
// One wave per (row, residue, column segment); lanes own columns.
__device__ __forceinline__ uint32_t window_bits(const Fr& k, uint32_t w, uint32_t c) {
    const uint32_t bit = w * c, limb = bit >> 5, sh = bit & 31;
    uint32_t lo = 0, hi = 0;
#pragma unroll
    for (int q = 0; q < 8; q++) {
        lo = (q == (int)limb) ? k.v[q] : lo;
        hi = (q == (int)limb + 1) ? k.v[q] : hi;
    }
    const uint64_t both = ((uint64_t)hi << 32) | lo;
    return (uint32_t)(both >> sh) & ((1u << c) - 1u);
}
// The bias H restricted to the bits a 256-bit word can hold: bit (c w + c - 1) for every window whose
// top bit lies below 256 (a window that reaches past bit 255 keeps its digit unsigned: see digit_of).
__device__ __forceinline__ Fr window_bias(uint32_t c, uint32_t nw) {
    Fr h = Fr::zero();
    for (uint32_t w = 0; w < nw; w++) {
        const uint32_t pos = w * c + c - 1;
#pragma unroll
        for (int i = 0; i < 8; i++) h.v[i] |= ((pos >> 5) == (uint32_t)i) ? (1u << (pos & 31)) : 0u;
    }
    return h;
}
// |k| + H for the half-range representative of a Montgomery-form scalar; flip = the scalar was negated.
// |k| <= (r-1)/2 < 0.91 * 2^254 and H < 1.01 * 2^255, so the sum stays below 2^256.
__device__ __forceinline__ Fr biased_half_range(const Fr& k_mont, const Fr& H, bool& flip) {
    Fr k = fr26::from_montc(k_mont);
    uint32_t borrow = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t half_i = (FrParams::mod(i) >> 1) | (i + 1 < 8 ? FrParams::mod(i + 1) << 31 : 0u);
        (void)detail::sbb32(half_i, k.v[i], borrow);
    }
    flip = borrow != 0;                                   // k > (r-1)/2
    k = cneg(k, flip);
    uint32_t carry = 0;
    Fr out;
#pragma unroll
    for (int i = 0; i < 8; i++) out.v[i] = detail::adc32(k.v[i], H.v[i], carry);
    return out;
}
// signed digit of window w of a biased scalar: in [-2^(c-1), 2^(c-1)) (unsigned, below 2^(256 - c w), for
// a top window whose bias bit does not exist)
__device__ __forceinline__ int32_t digit_of(const Fr& kb, uint32_t w, uint32_t c) {
    const int32_t bits = (int32_t)window_bits(kb, w, c);
    return (w * c + c - 1 < 256) ? bits - (int32_t)(1u << (c - 1)) : bits;
}

// acc += the windows q J + j, q0 <= q < q1, of k * G_col
__device__ __forceinline__ void madd_scalar_strided(Xyzz30& acc, const Fr& k_mont, const Fr& H, const uint32_t* table, size_t N, uint32_t col, uint32_t c,
                                                    uint32_t nw, uint32_t K, uint32_t J, uint32_t j, uint32_t q0, uint32_t q1) {
    bool flip;
    const Fr kb = biased_half_range(k_mont, H, flip);
    // digit of set q0 now, the next set's one addition ahead (its table line is touched early)
    int32_t d = q0 * J + j < nw ? digit_of(kb, q0 * J + j, c) : 0;
    uint32_t touch = 0;
    for (uint32_t q = q0; q < q1; q++) {
        const uint32_t wn = (q + 1) * J + j;
        const int32_t d_n = (q + 1 < q1 && wn < nw) ? digit_of(kb, wn, c) : 0;
        if (d != 0) {
            const bool neg = d < 0;
            const uint32_t mag = (uint32_t)(neg ? -d : d);
            const Affine30 e = ld_entry30(table, geom::table_entry(q, K, mag, N, col));
            const uint32_t mag_n = (uint32_t)(d_n < 0 ? -d_n : d_n);
            const size_t nxt = mag_n != 0 ? geom::table_entry(q + 1, K, mag_n, N, col) : (size_t)col;
            touch = table[(size_t)kWideEntryWords * nxt];
            if (kWideEntryWords % 32 != 0) touch |= table[(size_t)kWideEntryWords * nxt + kWideEntryWords - 1];
            madd30(acc, e, neg != flip);
        }
        d = d_n;
    }
    asm volatile("" ::"v"(touch));
}

__global__ void __launch_bounds__(kBlock) commit_strided_kernel(uint32_t* partial, const uint32_t* scalars, uint32_t rowlen, size_t rows,
                                                                uint32_t seg, uint32_t nseg, const uint32_t* table, size_t N,
                                                                uint32_t c, uint32_t nw, uint32_t K, uint32_t J, uint32_t nsets,
                                                                geom::WindowSplit split) {
    const int lane = threadIdx.x & 63;
    const size_t wave = ((size_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
    if (wave >= rows * J * nseg * split.parts) return;
    const size_t unit = wave / split.parts;
    const uint32_t q0 = (uint32_t)(wave - unit * split.parts) * split.per, q1 = q0 + split.per < nsets ? q0 + split.per : nsets;
    const geom::WaveSpan span = geom::wave_span(unit, nseg, seg, rowlen);   // "row" here is (row, residue)
    const size_t row = span.row / J;
    const uint32_t j = (uint32_t)(span.row - row * J);
    const Fr H = window_bias(c, nw);                      // wave-uniform
    Xyzz30 acc = xyzz30_inf();
    for (uint32_t col = span.s * seg + lane; col < span.col_end; col += 64)
        madd_scalar_strided(acc, ld_fr8(scalars, geom::scalar_index(row, rowlen, col)), H, table, N, col, c, nw, K, J, j, q0, q1);
    st_partial30(partial, wave * 64 + lane, acc);
}

// ------------------------------------------------------------------------------------------------
// commitment of the few elements of a tensor that a flag array lets through (full-width scalars)
// ------------------------------------------------------------------------------------------------
// G lanes per row, 64 / G rows per wave.  Every lane group sweeps its row's flags G columns at a
// time and queues the columns whose flag is zero in LDS; whenever some group has G queued (and once
// more at the end of the rows) every lane takes one queued column of its row, loads its scalar and
// adds scalar * G_col through the per-window table.  Lanes therefore work on dense batches however
// thinly the live elements are spread: sweeping the whole tensor with the dense kernel costs a
// recoding per element and an addition slot per WAVE that holds one live element - 80 ms for 2^27
// elements of which 0.7 % are live, against 3 ms here.  With many rows G = 32: a row of 4096 with
// 27 live elements fills 27 of 32 lanes of its batch instead of 27 of 64.
// With idx1 the scalars are table entries: element i is scalars[idx1[i] - 1].
__device__ __forceinline__ Fr ld_scalar(const uint32_t* scalars, const int32_t* __restrict__ idx1, size_t i) {
    if (!idx1) return ld_fr8(scalars, i);
    const uint32_t j = (uint32_t)idx1[i];
    return ld_fr8(scalars, j ? j - 1 : 0);
}
// The batch that ends a row deals shares of its columns' windows over the lanes: 27 live elements of a row and the larger of a
// wave's two rows decides (33 columns are two batches, half of the waves' lanes idle in the second).  2^27 elements of which
// 0.7 % are live, in rows of 4096: 3.77 -> 3.33 ms.
constexpr uint32_t kSparseShares = 5;
template <int G>
__global__ void __launch_bounds__(64) commit_sparse_fr_kernel(uint32_t* partial, const uint32_t* scalars, const int32_t* __restrict__ idx1,
                                                              const int32_t* __restrict__ skip, uint32_t rowlen, size_t rows, size_t step, const uint32_t* table, size_t N,
                                                              uint32_t c, uint32_t nw, uint32_t K, int* err_flag) {
    constexpr int R = 64 / G;                            // rows per wave
    __shared__ uint32_t queue[R][2 * G];
    const int lane = threadIdx.x;
    const int grp = lane / G, sub = lane % G;
    const size_t row = geom::spread_unit(blockIdx.x, gridDim.x, step) * R + grp;
    const bool have_row = row < rows;
    const unsigned long long gmask = (G == 64 ? ~0ull : ((1ull << (G & 63)) - 1ull)) << (grp * G);
    Xyzz30 acc = xyzz30_inf();
    uint32_t qn = 0;                                     // queued columns of this lane's row (uniform within the group)
    for (uint32_t base = 0;; base += G) {
        const bool last = base >= rowlen;
        if (!last) {
            const uint32_t col = base + sub;
            const bool take = have_row && col < rowlen && skip[geom::scalar_index(row, rowlen, col)] == 0;
            const unsigned long long m = __ballot(take) & gmask;
            if (take) queue[grp][qn + __popcll(m & ((1ull << lane) - 1ull))] = col;
            qn += (uint32_t)__popcll(m);
            __syncthreads();
        }
        // wave-uniform trigger: some group's batch is full, or the rows have ended with something queued
        const bool go = last ? __any(qn > 0) : __any(qn >= (uint32_t)G);
        if (go) {
            const uint32_t n = qn < (uint32_t)G ? qn : (uint32_t)G;
            // A full batch keeps every lane busy with a column of its own, the batch that ends a row does not: there a
            // lane takes a share of a column's windows, n * shares of them dealt over G lanes.
            const uint32_t units = last ? n * kSparseShares : n, per = last ? (nw + kSparseShares - 1) / kSparseShares : nw;
            for (uint32_t u = sub; u < units; u += G) {
                const uint32_t col = queue[grp][last ? u / kSparseShares : u], w0 = last ? (u % kSparseShares) * per : 0;
                const Fr k = from_mont(ld_scalar(scalars, idx1, geom::scalar_index(row, rowlen, col)));
                madd_scalar_fr(acc, k, table, N, col, c, nw, K, err_flag, w0, w0 + per);
            }
            __syncthreads();
            const uint32_t moved = (uint32_t)sub + G < qn ? queue[grp][sub + G] : 0u;
            __syncthreads();
            if ((uint32_t)sub + G < qn) queue[grp][sub] = moved;
            qn -= n;
            __syncthreads();
        }
        if (last) break;
    }
    if (have_row) st_partial30(partial, row * G + sub, acc);
}

// The same through the strided table: one wave per (row, residue) queues the row's live columns and works on them in
// batches of 64, so dead elements cost a look at their flag whether they lie scattered or in stretches, and a live one
// the strided table's 16 to 18 additions instead of the per-window table's 20.  Worth it from some hundred live elements a
// row (every residue leaves 64 partial sums).  One-wave workgroups, dealt by geom::spread_unit: the rows differ.
__global__ void __launch_bounds__(64) commit_sparse_strided_kernel(uint32_t* partial, const uint32_t* scalars, const int32_t* __restrict__ idx1,
                                                                   const int32_t* __restrict__ skip, uint32_t rowlen, size_t units, size_t step, const uint32_t* table, size_t N,
                                                                   uint32_t c, uint32_t nw, uint32_t K, uint32_t J, uint32_t nsets) {
    __shared__ uint32_t queue[2 * 64];
    const int lane = threadIdx.x;
    const size_t unit = geom::spread_unit(blockIdx.x, units, step), row = unit / J;
    const uint32_t j = (uint32_t)(unit - row * J);
    const Fr H = window_bias(c, nw);
    Xyzz30 acc = xyzz30_inf();
    uint32_t qn = 0;                                     // queued columns (uniform)
    for (uint32_t base = 0;; base += 64) {
        const bool last = base >= rowlen;
        if (!last) {
            const uint32_t col = base + lane;
            const bool take = col < rowlen && skip[geom::scalar_index(row, rowlen, col)] == 0;
            const unsigned long long m = __ballot(take);
            if (take) queue[qn + __popcll(m & ((1ull << lane) - 1ull))] = col;
            qn += (uint32_t)__popcll(m);
            __syncthreads();
        }
        if (qn >= 64 || (last && qn > 0)) {
            const uint32_t n = qn < 64 ? qn : 64;
            if ((uint32_t)lane < n) {
                const uint32_t col = queue[lane];
                madd_scalar_strided(acc, ld_scalar(scalars, idx1, geom::scalar_index(row, rowlen, col)), H, table, N, col, c, nw, K, J, j, 0, nsets);
            }
            __syncthreads();
            const uint32_t moved = (uint32_t)lane + 64 < qn ? queue[lane + 64] : 0u;
            __syncthreads();
            if ((uint32_t)lane + 64 < qn) queue[lane] = moved;
            qn -= n;
            __syncthreads();
        }
        if (last) break;
    }
    st_partial30(partial, unit * 64 + lane, acc);
}

// Row epilogue: the partial sums of a row become one point, the point its affine image.  Three kernels:
//   commit_reduce_lane_kernel  rows by the ten thousand: one lane per kept partial sum adds its share (88 wave
//                              instructions per addition, the fewest, but chains of 7 additions at 15 us each)
//   commit_reduce_quad_kernel  2^lg_qpr quads (quad30.hpp) per row, each adds its share, then a tree of shuffles
//                              (140 wave instructions per addition, 4.8 us each)
//   quad_affine_kernel         the map to affine coordinates, a quad per row
// geom::reduce_plan picks.  Bound: instruction latency - a SIMD issues hardly faster with two of these waves than with
// one, so what counts is one wave per SIMD (workgroups of four waves spread evenly over a compute unit's
// SIMDs, one-wave workgroups do not: 139 against 175 us for 4096 rows of 64) and few additions in a chain.
// The map is a kernel of its own so that every quad of a wave inverts: left to the sum kernel's first quads
// it took 0.1 ms longer.  Measured, one box, before (one lane per accumulator, shuffle or LDS trees) and now:
// 4096 rows of 64: 0.291 -> 0.148 ms (0.136 on 13 limbs); 512 of 64: 0.196 -> 0.079; one of 4096: 0.277 -> 0.124; 64 of 256: 0.237 -> 0.093;
// 32768 of 64: 1.08 -> 0.54.
__device__ __forceinline__ quad::Acc ld_quad_partial(const uint32_t* base, size_t i) {
    const uint32_t* p = base + geom::partial_word(i);
    const uint2* q = reinterpret_cast<const uint2*>(p + (threadIdx.x & 3) * kCoordWords);
    uint2 w[kCoordWords / 2];
#pragma unroll
    for (int k = 0; k < kCoordWords / 2; k++) w[k] = q[k];
    const uint32_t* f = reinterpret_cast<const uint32_t*>(w);
    quad::Acc a;
#pragma unroll
    for (int k = 0; k < L30; k++) a.v.v[k] = (int32_t)f[k];
    a.inf = p[4 * kCoordWords] != 0;
    return a;
}
__device__ __forceinline__ void st_quad_partial(uint32_t* base, size_t i, const quad::Acc& a) {
    uint32_t* p = base + geom::partial_word(i);
    uint2* q = reinterpret_cast<uint2*>(p + (threadIdx.x & 3) * kCoordWords);
    uint32_t f[kCoordWords];
#pragma unroll
    for (int k = 0; k < kCoordWords; k++) f[k] = k < L30 ? (uint32_t)a.v.v[k] : 0u;
#pragma unroll
    for (int k = 0; k < kCoordWords / 2; k++) q[k] = make_uint2(f[2 * k], f[2 * k + 1]);
    if ((threadIdx.x & 3) == 0) p[4 * kCoordWords] = a.inf ? 1u : 0u;
}
__global__ void __launch_bounds__(kBlock) commit_reduce_quad_kernel(uint32_t* out, const uint32_t* partial, size_t rows, uint32_t nparts,
                                                                    uint32_t lg_qpr) {
    const int lane = threadIdx.x & 63;
    const size_t wave = ((size_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
    const uint32_t qpr = 1u << lg_qpr, sub = geom::quad_share(lane, lg_qpr);
    const size_t row = geom::reduce_row(wave, lane, lg_qpr + 2);
    const bool have = row < rows;
    quad::Acc acc = quad::identity(), next = quad::identity();
    const uint32_t nserial = (nparts + qpr - 1) >> lg_qpr;
    if (have && sub < nparts) next = ld_quad_partial(partial, row * nparts + sub);
    // one addition site serves both the serial part and the tree steps (code size); the next partial sum is on its way
    // while this one is added
    for (uint32_t step = 0; step < nserial + lg_qpr; step++) {
        quad::Acc q = next;
        next = quad::identity();
        if (step < nserial) {
            const uint32_t j = sub + ((step + 1) << lg_qpr);
            if (have && j < nparts) next = ld_quad_partial(partial, row * nparts + j);
        } else {
            const uint32_t off = (qpr >> 1) >> (step - nserial);
#pragma unroll
            for (int k = 0; k < L30; k++) q.v.v[k] = __shfl_down(acc.v.v[k], 4 * off, 64);
            q.inf = __shfl_down((int)acc.inf, 4 * off, 64) != 0 || sub + off >= qpr;
        }
        quad::add(acc, q);
    }
    if (have && sub == 0) st_quad_partial(out, row, acc);      // 256 bytes per row: an accumulator
}
template <bool START>
__global__ void __launch_bounds__(kBlock) quad_affine_kernel(uint32_t* out, const uint32_t* sums, size_t rows, const uint32_t* start) {
    const size_t row = ((size_t)blockIdx.x * kBlock + threadIdx.x) >> 2;
    if (row >= rows) return;
    quad::Acc acc = ld_quad_partial(sums, row);
    if (START) quad::add(acc, ld_quad_partial(start, 0));
    const Fp c = quad::to_affine(acc);
    const uint32_t r = threadIdx.x & 3;
    if (r < 2) st_fp(out + 2 * FW * row + FW * r, c);
}
// out[row] = sum_j 2^(c j) A[row * J + j] by Horner from the top residue or window down, then affine: a chain of (J - 1) c
// doublings, so a quad per row (three products' time a doubling, where one lane runs nine products.
// One row of 32 byte windows, 248 doublings: 6.6 -> 1.1 ms; four residues of 16 bits, 48 doublings: 0.54 -> 0.26 ms).
__global__ void __launch_bounds__(64) quad_horner_kernel(uint32_t* out, const uint32_t* sums, size_t rows, uint32_t J, uint32_t c) {
    const size_t row = ((size_t)blockIdx.x * 64 + threadIdx.x) >> 2;
    if (row >= rows) return;
    quad::Acc total = ld_quad_partial(sums, row * J + (J - 1));
    for (int j = (int)J - 2; j >= 0; j--) {
        for (uint32_t d = 0; d < c; d++) quad::dbl(total);
        quad::add(total, ld_quad_partial(sums, row * J + j));
    }
    const Fp v = quad::to_affine(total);
    const uint32_t r = threadIdx.x & 3;
    if (r < 2) st_fp(out + 2 * FW * row + FW * r, v);
}
// out[row * keep + k] = the sum of the row's partial sums k, k + keep, ...
__global__ void __launch_bounds__(kBlock) commit_reduce_lane_kernel(uint32_t* out, const uint32_t* partial, size_t rows, uint32_t nparts, uint32_t keep) {
    const size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (t >= rows * keep) return;
    const size_t row = geom::lane_row(t, keep);
    const uint32_t sub = geom::lane_share(t, keep);
    Xyzz30 acc = ld_partial30(partial, row * nparts + sub);
    for (uint32_t j = sub + keep; j < nparts; j += keep) padd30(acc, ld_partial30(partial, row * nparts + j));
    st_partial30(out, t, acc);
}

// ------------------------------------------------------------------------------------------------
// sum_i k_i P_i over arbitrary points (the row commitments of a verification: no table of multiples exists).
// Signed 4-bit windows: the multiples P, 2P .. 8P of every point, then for each of the 64 windows w the sum
// S_w = sum_i digit_w(k_i) P_i, everything on quads - a few hundred points are a latency problem, and the only long
// chain, sum_w 16^w S_w with its 252 doublings, is left to the host, whose core runs a doubling in 0.8 us where a lone
// quad takes 4.  256 points: 0.1 ms against 200 ms for 255 scalar multiples on the host.
// ------------------------------------------------------------------------------------------------
constexpr uint32_t kMsmWindows = GRAPE_MSM_WINDOWS, kMsmBits = 4, kMsmMultiples = 1u << (kMsmBits - 1);
constexpr uint32_t kMsmGroup = 64;             // points that one wave sums
// table[i * 8 + k - 1] = k P_i, a quad per entry
__global__ void __launch_bounds__(kBlock) msm_multiples_kernel(uint32_t* table, const uint32_t* points, size_t n) {
    const size_t q = ((size_t)blockIdx.x * kBlock + threadIdx.x) >> 2;
    if (q >= n * kMsmMultiples) return;
    const uint32_t k = (uint32_t)(q % kMsmMultiples) + 1;
    const int r = threadIdx.x & 3;
    const Fp w = ld_fp(points + 3 * FW * (q / kMsmMultiples) + FW * (r < 2 ? r : 2));     // x, y, z, z
    quad::Acc p;
    p.inf = quad::perm<quad::ctrl(2, 2, 2, 2)>((int32_t)w.is_zero()) != 0;
    const Fp30 v = fp30::from_canonical_lazy(w);
    const Fp30 zz = fp30::sqr(v);
    p.v = quad::select(quad::lanes<0>() | quad::lanes<1>(), v, quad::select(quad::lanes<2>(), zz, fp30::mul(zz, v)));
    quad::Acc acc = p;
    for (int b = 30 - __clz((int)k); b >= 0; b--) {
        quad::dbl(acc);
        if ((k >> b) & 1) quad::add(acc, p);
    }
    st_quad_partial(table, q, acc);
}
// partial[w * stride + g] = the sum of window w's digits times the points of group g
__global__ void __launch_bounds__(kBlock) msm_window_kernel(uint32_t* partial, const uint32_t* table, const uint32_t* scalars, size_t n,
                                                            uint32_t groups, size_t stride) {
    const int lane = threadIdx.x & 63;
    const size_t unit = ((size_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
    const uint32_t w = (uint32_t)(unit / groups), g = (uint32_t)(unit % groups);
    if (w >= kMsmWindows) return;
    const Fr H = window_bias(kMsmBits, kMsmWindows);
    const uint32_t sub = (uint32_t)lane >> 2;
    quad::Acc acc = quad::identity();
    constexpr uint32_t kSerial = kMsmGroup / 16;
    for (uint32_t step = 0; step < kSerial + 4; step++) {
        quad::Acc q = quad::identity();
        if (step < kSerial) {
            const size_t i = (size_t)g * kMsmGroup + step * 16 + sub;
            if (i < n) {
                bool flip;
                const int32_t d = digit_of(biased_half_range(ld_fr8(scalars, i), H, flip), w, kMsmBits);
                if (d != 0) {
                    q = ld_quad_partial(table, i * kMsmMultiples + (uint32_t)(d < 0 ? -d : d) - 1);
                    quad::cneg(q, (d < 0) != flip);
                }
            }
        } else {
            const uint32_t off = 8u >> (step - kSerial);
#pragma unroll
            for (int k = 0; k < L30; k++) q.v.v[k] = __shfl_down(acc.v.v[k], 4 * off, 64);
            q.inf = __shfl_down((int)acc.inf, 4 * off, 64) != 0 || sub + off >= 16;
        }
        quad::add(acc, q);
    }
    if (sub == 0) st_quad_partial(partial, (size_t)w * stride + g, acc);
}
// accumulators in the working form -> XYZZ points in the memory form, a lane per coordinate
__global__ void __launch_bounds__(64) quad_canonical_kernel(uint32_t* out, const uint32_t* sums, size_t n) {
    const size_t q = ((size_t)blockIdx.x * 64 + threadIdx.x) >> 2;
    if (q >= n) return;
    const quad::Acc a = ld_quad_partial(sums, q);
    st_fp(out + 4 * FW * q + FW * (threadIdx.x & 3), a.inf ? Fp::zero() : fp30::to_canonical(a.v));
}

// ------------------------------------------------------------------------------------------------
// commitment through the reference-format table (entry k * npoints + i = k * G_i, k < 256, canonical
// affine points): the reference's algorithm (byte windows, 8 doublings between windows,
// src/Hyrax.cu:46-167) re-ordered so that it fills the chip whatever the number of rows - one wave
// per (row, window, column segment) sums its table entries in the working form, the row-reduction
// kernel folds the lanes and segments of every (row, window), and a last kernel runs the Horner
// chain over a row's windows.  A table entry is converted on the fly (one product per
// coordinate); no wide table has to be built, which is what single rows (Hyrax::open's blinding
// row, single_commit) and rows too long for a wide table need.
// ------------------------------------------------------------------------------------------------
template <bool FR>
__global__ void __launch_bounds__(kBlock, 2) commit_ref30_kernel(uint32_t* partial, const void* scalars, uint32_t rowlen, size_t rows,
                                                                 uint32_t seg, uint32_t nseg, const uint32_t* table, size_t npoints) {
    constexpr uint32_t nwin = FR ? 32 : 4;
    const size_t unit = ((size_t)blockIdx.x * kBlock + threadIdx.x) >> 6;      // one wave per unit
    const uint32_t lane = threadIdx.x & 63;
    if (unit >= rows * nwin * nseg) return;
    const uint32_t sg = (uint32_t)(unit % nseg);
    const size_t rw = unit / nseg;
    const uint32_t w = (uint32_t)(rw % nwin);
    const size_t row = rw / nwin;
    const uint32_t col_end = (sg + 1) * seg < rowlen ? (sg + 1) * seg : rowlen;
    Xyzz30 acc = xyzz30_inf();
    for (uint32_t col = sg * seg + lane; col < col_end; col += 64) {
        uint32_t idx;
        bool neg = false;
        if (FR) {
            const Fr k = fr26::from_montc(ld_fr8((const uint32_t*)scalars, row * rowlen + col));
            uint32_t limb = 0;
#pragma unroll
            for (int q = 0; q < 8; q++) limb = (q == (int)(w >> 2)) ? k.v[q] : limb;
            idx = (limb >> (8 * (w & 3))) & 255u;
        } else {
            const int32_t sv = ((const int32_t*)scalars)[row * rowlen + col];
            neg = sv < 0;
            const uint32_t a = neg ? (uint32_t)0 - (uint32_t)sv : (uint32_t)sv;
            idx = (a >> (8 * w)) & 255u;
        }
        if (idx) {
            const G1Affine a = ld_affine(table, (size_t)idx * npoints + col);
            if (!a.is_inf()) {
                Affine30 e;
                e.x = fp30::from_canonical_lazy(a.x);
                e.y = fp30::from_canonical_lazy(a.y);
                if (!xyzz30_madd(acc, e, neg)) {           // entry = +-accumulator: exact canonical-form addition
                    G1Xyzz c = xyzz30_to_canonical(acc);
                    xyzz_add_affine(c, a, neg);
                    acc = xyzz30_from_canonical(c);
                }
            }
        }
    }
    st_partial30(partial, unit * 64 + lane, acc);
}

__global__ void __launch_bounds__(64) affine_to_jac_kernel(uint32_t* out, const uint32_t* in, size_t n) {
    size_t i = (size_t)blockIdx.x * 64 + threadIdx.x;
    if (i >= n) return;
    G1Affine a = ld_affine(in, i);
    bool inf = a.is_inf();
    st_fp(out + 3 * FW * i, a.x);
    st_fp(out + 3 * FW * i + FW, a.y);
    st_fp(out + 3 * FW * i + 2 * FW, inf ? Fp::zero() : Fp::one());
}
__global__ void __launch_bounds__(64) jac_to_affine_kernel(uint32_t* out, const uint32_t* in, size_t n) {
    size_t i = (size_t)blockIdx.x * 64 + threadIdx.x;
    if (i >= n) return;
    G1Jac p;
    p.x = ld_fp(in + 3 * FW * i);
    p.y = ld_fp(in + 3 * FW * i + FW);
    p.z = ld_fp(in + 3 * FW * i + 2 * FW);
    G1Affine a = G1Affine::inf();
    if (!p.is_inf()) {
        const Fp zi = fp_inverse_fast(p.z), zi2 = fsqr(zi);
        a.x = fmul(p.x, zi2);
        a.y = fmul(p.y, fmul(zi2, zi));
    }
    st_affine(out, i, a);
}

// out[i] = a[i] + b[i] for affine points (either may be the point at infinity, or both equal or opposite)
__global__ void __launch_bounds__(64) affine_add_kernel(uint32_t* out, const uint32_t* a, const uint32_t* b, size_t n) {
    size_t i = (size_t)blockIdx.x * 64 + threadIdx.x;
    if (i >= n) return;
    G1Xyzz acc = G1Xyzz::inf();
    madd(acc, ld_affine(a, i), false);
    madd(acc, ld_affine(b, i), false);
    st_affine(out, i, to_affine(acc));
}

}  // namespace grape

using namespace grape;

#define CHECK_PTR16(p) GRAPE_REQUIRE((p) != nullptr && (reinterpret_cast<uintptr_t>(p) & 15) == 0, #p " must be a 16-byte aligned device pointer")

using geom::reduce_lanes_log2;
// Largest commitment one call accepts: 2^28 scalars (1 GiB of int32, 8 GiB of field elements), the
// largest size the GPU tests run; the host classes split longer tensors by rows.
constexpr size_t kMaxCommitScalars = (size_t)1 << 28;

// Row reduction of `rows` rows of `nparts` partial sums each (`tmp`: work space of reduce_tmp_bytes): to affine points, or
// to accumulators of 256 bytes for a later combination.
static size_t reduce_tmp_bytes(size_t rows, uint32_t nparts) { return geom::reduce_tmp_accumulators(rows, nparts) * (4 * kPartialWords); }
template <bool AFFINE>
static void launch_reduce(uint32_t* out, const uint32_t* partial, size_t rows, uint32_t nparts, uint32_t* tmp, hipStream_t s, const uint32_t* start = nullptr) {
    geom::ReduceStage st[geom::kMaxReduceStages];
    const int n = geom::reduce_stages(rows, nparts, st);
    uint32_t* sums = nullptr;
    for (int i = 0; i < n; i++) {
        const uint32_t* from = i == 0 ? partial : tmp + geom::partial_word(st[i].from);
        sums = i == n - 1 && !AFFINE ? out : tmp + geom::partial_word(st[i].to);
        if (st[i].lanes) commit_reduce_lane_kernel<<<blocks_for(st[i].units * st[i].keep), kBlock, 0, s>>>(sums, from, st[i].units, st[i].parts, st[i].keep);
        else commit_reduce_quad_kernel<<<blocks_for(st[i].units << (st[i].lg_qpr + 2)), kBlock, 0, s>>>(sums, from, st[i].units, st[i].parts, st[i].lg_qpr);
    }
    if (AFFINE && start) quad_affine_kernel<true><<<blocks_for(rows * 4), kBlock, 0, s>>>(out, sums, rows, start);
    else if (AFFINE) quad_affine_kernel<false><<<blocks_for(rows * 4), kBlock, 0, s>>>(out, sums, rows, nullptr);
}

template <bool FR>
static int commit_wide_impl(uint32_t* out, const void* scalars, size_t size, uint32_t rowlen, const uint32_t* table, size_t N,
                            uint32_t c, uint32_t nw, uint32_t K, grape_stream_t st, int* caller_flag = nullptr, const CommitBase* base = nullptr) {
    if (size == 0) return GRAPE_OK;                      // no rows: nothing is read or written
    GRAPE_REQUIRE(size <= kMaxCommitScalars, "more than 2^28 scalars in one call: commit the rows in several calls");
    CHECK_PTR16(out); CHECK_PTR16(scalars); CHECK_PTR16(table);
    GRAPE_REQUIRE(rowlen >= 1 && size % rowlen == 0, "size must be a multiple of rowlen");
    GRAPE_REQUIRE(rowlen <= N, "row longer than the generator set");
    // a single-window table may hold fewer than 2^(c-1) multiples (the indexed commitments: K table
    // rows, digits 1..K); a digit above K is caught on the device
    GRAPE_REQUIRE(c >= 2 && c <= (FR ? 16u : 24u) && nw >= 1 && K >= 1 && (K >= (1u << (c - 1)) || (!FR && nw == 1)),
                  "need 2 <= c <= 16 (24 for int32) and K >= 2^(c-1) (any K >= 1 with one window of int32 digits)");
    if (FR) GRAPE_REQUIRE((uint64_t)nw * c >= 255, "Fr scalars need nw*c >= 255");
    const size_t rows = size / rowlen;
    if (rows == 0) return GRAPE_OK;
    hipStream_t s = as_stream(st);
    // rows go through in slabs so that the per-lane partial sums stay within 512 MiB whatever the
    // number of rows (a row segment leaves 64 partial sums of 256 bytes)
    const geom::WidePlan plan = geom::wide_plan(size, rowlen, geom::kSlabSegments);
    const uint32_t nseg = plan.nseg, seg = plan.seg;
    geom::WindowSplit split = {1, nw};
    if (FR) split = geom::window_split(rows * nseg, nw);
    const uint32_t nparts = nseg * split.parts * 64;
    const size_t slab = plan.slab, partial_bytes = plan.partial_bytes * split.parts;
    void* ws;
    const size_t tmp_bytes = reduce_tmp_bytes(slab, nparts);
    int rc = scratch_get(kSlotMsm, partial_bytes + tmp_bytes + 64, &ws, s);
    if (rc) return rc;
    uint32_t* red_tmp = (uint32_t*)((char*)ws + partial_bytes);
    // the digit-range flag: the call's own (cleared here, read back at the end), or one the caller
    // owns, has cleared and reads when it likes - then nothing here waits for the stream
    int* err = caller_flag ? caller_flag : (int*)((char*)ws + partial_bytes + tmp_bytes);
    if (!caller_flag) {
        rc = zero_fill(err, sizeof(int), s);
        if (rc) return rc;
    }
    const size_t elem_words = FR ? 8 : 1;
    profile_begin();
    for (size_t r0 = 0; r0 < rows; r0 += slab) {
        const size_t nr = rows - r0 < slab ? rows - r0 : slab;
        const uint32_t* sc = (const uint32_t*)scalars + r0 * rowlen * elem_words;
        profile_mark(s);
        if (!FR && base) {
            const size_t waves = nr * nseg, step = base->step ? geom::spread_step(waves) : 0;
            commit_wide_kernel<false, true><<<step ? (unsigned)waves : blocks_for(nr * nparts), step ? 64 : kBlock, 0, s>>>(
                (uint32_t*)ws, sc, rowlen, nr, seg, nseg, table, N, c, nw, K, err, split, CommitBase{base->start, base->base1, step});
        } else
            commit_wide_kernel<FR><<<blocks_for(nr * nparts), kBlock, 0, s>>>((uint32_t*)ws, sc, rowlen, nr, seg, nseg, table, N, c, nw, K, err, split, CommitBase{});
        profile_mark(s);
        launch_reduce<true>(out + r0 * (size_t)(2 * FW), (const uint32_t*)ws, nr, nparts, red_tmp, s, base ? base->start : nullptr);
        profile_mark(s);
    }
    GRAPE_LAUNCH_CHECK();
    if (caller_flag) return GRAPE_OK;
    int h_err = 0;
    GRAPE_HIP_CHECK(hipMemcpyAsync(&h_err, err, sizeof(int), hipMemcpyDeviceToHost, s));
    GRAPE_HIP_CHECK(hipStreamSynchronize(s));
    if (h_err) {
        set_error("commit: a scalar does not fit the table's digit range (c=%u, nw=%u, K=%u)", c, nw, K);
        return GRAPE_EINVAL;
    }
    return GRAPE_OK;
}

template <bool FR>
static int commit_ref_impl(uint32_t* out, const void* scalars, size_t size, uint32_t rowlen, const uint32_t* table, size_t npoints,
                           grape_stream_t st) {
    if (size == 0) return GRAPE_OK;                      // no rows: nothing is read or written
    GRAPE_REQUIRE(size <= kMaxCommitScalars, "more than 2^28 scalars in one call: commit the rows in several calls");
    CHECK_PTR16(out); CHECK_PTR16(scalars); CHECK_PTR16(table);
    GRAPE_REQUIRE(rowlen >= 1 && size % rowlen == 0 && rowlen <= npoints, "bad shape");
    const size_t rows = size / rowlen;
    if (rows == 0) return GRAPE_OK;
    hipStream_t s = as_stream(st);
    const uint32_t nwin = FR ? 32 : 4;
    // column segments: enough waves to fill the chip, at least one 64-column sweep each, and chains
    // of at most 128 partial sums per reducing lane
    const uint32_t lg_lpr = reduce_lanes_log2(rows * nwin);
    uint32_t nseg = 1;
    while (rows * nwin * nseg < 8192 && rowlen / (nseg * 2) >= 64 && nseg * 2 <= (2u << lg_lpr)) nseg *= 2;
    const uint32_t seg = (rowlen + nseg - 1) / nseg;
    // rows go through in slabs so that the per-lane partial sums stay within 512 MiB
    size_t slab = 32768 / ((size_t)nwin * nseg);
    if (slab < 1) slab = 1;
    if (slab > rows) slab = rows;
    const size_t partial_bytes = slab * nwin * nseg * 64 * (size_t)(4 * kPartialWords);
    void* ws;
    const size_t sums_bytes = slab * nwin * (size_t)(4 * kPartialWords);
    int rc = scratch_get(kSlotMsm, partial_bytes + sums_bytes + reduce_tmp_bytes(slab * nwin, nseg * 64) + 64, &ws, s);
    if (rc) return rc;
    uint32_t* sums = (uint32_t*)((char*)ws + partial_bytes);
    uint32_t* red_tmp = (uint32_t*)((char*)ws + partial_bytes + sums_bytes);
    const size_t elem_words = FR ? 8 : 1;
    for (size_t r0 = 0; r0 < rows; r0 += slab) {
        const size_t nr = rows - r0 < slab ? rows - r0 : slab;
        const size_t units = nr * nwin * nseg;
        const uint32_t* sc = (const uint32_t*)scalars + r0 * rowlen * elem_words;
        commit_ref30_kernel<FR><<<blocks_for(units * 64), kBlock, 0, s>>>((uint32_t*)ws, sc, rowlen, nr, seg, nseg, table, npoints);
        launch_reduce<false>(sums, (const uint32_t*)ws, nr * nwin, nseg * 64, red_tmp, s);
        quad_horner_kernel<<<blocks_for(nr * 4, 64), 64, 0, s>>>(out + r0 * (size_t)(2 * FW), sums, nr, nwin, 8);
    }
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

extern "C" {

int grape_g1_generator(uint32_t* out) {
    GRAPE_REQUIRE(out != nullptr, "null output");
    for (int i = 0; i < FW; i++) {
        out[i] = g1_gen_x(i);
        out[FW + i] = g1_gen_y(i);
    }
    return GRAPE_OK;
}

int grape_g1_scalar_mul_base(uint32_t* out, const uint32_t* k, const uint32_t* base, size_t n, grape_stream_t st) {
    if (n == 0) return GRAPE_OK;
    CHECK_PTR16(out); CHECK_PTR16(k); CHECK_PTR16(base);
    scalar_mul_base_kernel<<<blocks_for(n, 64), 64, 0, as_stream(st)>>>(out, k, base, n);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

static int wide_table_gen_impl(uint32_t* table, const uint32_t* gens, size_t N, uint32_t c, uint32_t nw, uint32_t K, grape_stream_t st);

// The multiples come from the level-wise generator of the wide tables (one window, K = W - 1), a
// slab of generators at a time through a staging table of at most 1 GiB, and are then rewritten in
// the reference's layout and limb form.
int grape_g1_table_gen(uint32_t* table, const uint32_t* gens, size_t N, uint32_t W, grape_stream_t st) {
    if (N == 0 || W == 0) return GRAPE_OK;
    CHECK_PTR16(table); CHECK_PTR16(gens);
    GRAPE_REQUIRE(W <= (1u << 16), "bad table shape");
    hipStream_t s = as_stream(st);
    const uint32_t K = W > 1 ? W - 1 : 1;
    size_t slab = ((size_t)1 << 30) / ((size_t)K * 4 * kWideEntryWords);
    if (slab < 64) slab = 64;
    if (slab > N) slab = N;
    void* stage;
    int rc = scratch_get(kSlotTable, slab * K * 4 * kWideEntryWords, &stage, s);
    if (rc) return rc;
    for (size_t i0 = 0; i0 < N; i0 += slab) {
        const size_t ns = N - i0 < slab ? N - i0 : slab;
        if (W > 1) {
            rc = wide_table_gen_impl((uint32_t*)stage, gens + i0 * (size_t)(2 * FW), ns, 1, 1, K, st);
            if (rc) return rc;
        }
        ref_from_wide_kernel<<<blocks_for(ns * W), kBlock, 0, s>>>(table, (const uint32_t*)stage, N, i0, ns, W);
        GRAPE_LAUNCH_CHECK();
    }
    return GRAPE_OK;
}

size_t grape_g1_wide_table_bytes(size_t N, uint32_t nw, uint32_t K) { return (size_t)nw * K * N * 4 * kWideEntryWords; }

// table[(w*K + k-1)*N + i] = k * 2^(spacing*w) * G_i for k = 1..K, w < nw
static int wide_table_gen_impl(uint32_t* table, const uint32_t* gens, size_t N, uint32_t c, uint32_t nw, uint32_t K, grape_stream_t st) {
    hipStream_t s = as_stream(st);
    const size_t per_chunk = (size_t)nw * N;
    // the first CH multiples of every base as a chain of mixed additions, normalised together;
    // everything above them level by level from the entries below (wide_extend_kernel)
    uint32_t CH = kFirstChain;
    if (K < CH) CH = K;
    void* ws;
    const size_t bases_bytes = per_chunk * (8 * FW);
    const size_t tmp_bytes = (size_t)CH * per_chunk * (16 * FW);
    int rc = scratch_get(kSlotMsm, bases_bytes + tmp_bytes + 256, &ws, s);
    if (rc) return rc;
    uint32_t* bases = (uint32_t*)ws;
    uint32_t* tmp = (uint32_t*)((char*)ws + bases_bytes);
    int* degenerate = (int*)((char*)ws + bases_bytes + tmp_bytes);
    rc = zero_fill(degenerate, sizeof(int), s);
    if (rc) return rc;
    window_bases_kernel<<<blocks_for(N, 64), 64, 0, s>>>(bases, gens, N, c, nw);
    GRAPE_LAUNCH_CHECK();
    {
        wide_chain_kernel<<<blocks_for(per_chunk, 64), 64, 0, s>>>(tmp, bases, N, nw, K, CH, 0, 1);
        const size_t n_entries = (size_t)CH * per_chunk;
        const size_t nthr2 = (n_entries + kNormChunk - 1) / kNormChunk;
        wide_normalize_kernel<<<blocks_for(nthr2, 64), 64, 0, s>>>(table, tmp, N, nw, K, CH, 0, n_entries);
        GRAPE_LAUNCH_CHECK();
    }
    for (uint32_t have = CH; have < K;) {
        const uint32_t cnt = K - have < have ? K - have : have;
        const uint32_t run = cnt < kExtendRun ? cnt : kExtendRun;
        const size_t nthreads = per_chunk * ((cnt + run - 1) / run);
        const size_t exact_want = (per_chunk * cnt + 63) / 64;
        const unsigned exact_blocks = (unsigned)(exact_want < 16384 ? exact_want : 16384);   // a no-op unless the flag is up
        wide_extend_kernel<<<blocks_for(nthreads), kBlock, 0, s>>>(table, N, nw, K, have, cnt, run, degenerate);
        wide_extend_exact_kernel<<<exact_blocks, 64, 0, s>>>(table, N, nw, K, have, cnt, degenerate);
        GRAPE_LAUNCH_CHECK();
        have += cnt;
    }
    return GRAPE_OK;
}

int grape_g1_wide_table_gen(uint32_t* table, const uint32_t* gens, size_t N, uint32_t c, uint32_t nw, uint32_t K, grape_stream_t st) {
    CHECK_PTR16(table); CHECK_PTR16(gens);
    GRAPE_REQUIRE(N >= 1 && c >= 1 && c <= 16 && nw >= 1 && K >= 1 && K <= (1u << 16), "bad table shape");
    return wide_table_gen_impl(table, gens, N, c, nw, K, st);
}

int grape_g1_strided_table_gen(uint32_t* table, const uint32_t* gens, size_t N, uint32_t c, uint32_t J, uint32_t nsets, grape_stream_t st) {
    CHECK_PTR16(table); CHECK_PTR16(gens);
    GRAPE_REQUIRE(N >= 1 && c >= 2 && c <= 18 && J >= 1 && nsets >= 1 && (uint64_t)c * J * (nsets - 1) < 256, "bad table shape");
    return wide_table_gen_impl(table, gens, N, c * J, nsets, 1u << (c - 1), st);
}

// Full-width scalars through a strided table (see commit_strided_kernel): nw = ceil(255 / c) windows,
// J residues, nsets = ceil(nw / J) table sets of K = 2^(c-1) multiples.
static int commit_strided_impl(uint32_t* out, const uint32_t* scalars, const int32_t* idx1, const int32_t* skip, size_t size, uint32_t rowlen, const uint32_t* table,
                               size_t N, uint32_t c, uint32_t J, uint32_t nsets, grape_stream_t st) {
    if (size == 0) return GRAPE_OK;
    GRAPE_REQUIRE(size <= kMaxCommitScalars, "more than 2^28 scalars in one call: commit the rows in several calls");
    CHECK_PTR16(out); CHECK_PTR16(scalars); CHECK_PTR16(table);
    GRAPE_REQUIRE(rowlen >= 1 && size % rowlen == 0, "size must be a multiple of rowlen");
    GRAPE_REQUIRE(rowlen <= N, "row longer than the generator set");
    GRAPE_REQUIRE(c >= 2 && c <= 18 && J >= 1, "need 2 <= c <= 18 and J >= 1");
    const uint32_t nw = (255 + c - 1) / c, K = 1u << (c - 1);
    GRAPE_REQUIRE(J <= nw && (uint64_t)nsets * J >= nw, "nsets * J must cover ceil(255 / c) windows");
    const size_t rows = size / rowlen;
    hipStream_t s = as_stream(st);
    // (row, residue) pairs are the rows of the accumulation and reduction launches
    const geom::WidePlan plan = geom::wide_plan(rows * J * (size_t)rowlen, rowlen, geom::kSlabSegments);
    const uint32_t nseg = skip ? 1 : plan.nseg, seg = plan.seg;      // with flags a wave takes a whole row
    size_t slab = (skip ? geom::kSlabSegments : plan.slab) / J;                              // whole rows per launch
    if (slab < 1) slab = 1;
    if (slab > rows) slab = rows;
    geom::WindowSplit split = {1, nsets};
    if (!skip) split = geom::window_split(rows * J * nseg, nsets);
    const uint32_t nparts = nseg * split.parts * 64;
    const size_t partial_bytes = slab * J * nparts * (size_t)(4 * kPartialWords);
    const size_t sums_bytes = slab * J * (size_t)(4 * kPartialWords);
    void* ws;
    int rc = scratch_get(kSlotMsm, partial_bytes + sums_bytes + reduce_tmp_bytes(slab * J, nparts), &ws, s);
    if (rc) return rc;
    uint32_t* sums = (uint32_t*)((char*)ws + partial_bytes);
    uint32_t* red_tmp = (uint32_t*)((char*)ws + partial_bytes + sums_bytes);
    profile_begin();
    for (size_t r0 = 0; r0 < rows; r0 += slab) {
        const size_t nr = rows - r0 < slab ? rows - r0 : slab;
        const uint32_t* sc = idx1 ? scalars : scalars + r0 * rowlen * 8;
        profile_mark(s);
        if (skip)
            commit_sparse_strided_kernel<<<(unsigned)(nr * J), 64, 0, s>>>((uint32_t*)ws, sc, idx1 ? idx1 + r0 * rowlen : nullptr, skip + r0 * rowlen, rowlen, nr * J, geom::spread_step(nr * J),
                                                                           table, N, c, nw, K, J, nsets);
        else
            commit_strided_kernel<<<blocks_for(nr * J * nparts), kBlock, 0, s>>>((uint32_t*)ws, sc, rowlen, nr, seg, nseg, table, N, c, nw, K, J, nsets, split);
        profile_mark(s);
        launch_reduce<false>(sums, (const uint32_t*)ws, nr * J, nparts, red_tmp, s);
        quad_horner_kernel<<<blocks_for(nr * 4, 64), 64, 0, s>>>(out + r0 * (size_t)(2 * FW), sums, nr, J, c);
        profile_mark(s);
    }
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

int grape_commit_fr_strided(uint32_t* out, const uint32_t* scalars, size_t size, uint32_t rowlen, const uint32_t* table, size_t N,
                            uint32_t c, uint32_t J, uint32_t nsets, grape_stream_t st) {
    return commit_strided_impl(out, scalars, nullptr, nullptr, size, rowlen, table, N, c, J, nsets, st);
}
int grape_commit_fr_strided_masked(uint32_t* out, const uint32_t* scalars, const int32_t* skip, size_t size, uint32_t rowlen, const uint32_t* table,
                                   size_t N, uint32_t c, uint32_t J, uint32_t nsets, grape_stream_t st) {
    GRAPE_REQUIRE(size == 0 || skip != nullptr, "no flag array");
    return commit_strided_impl(out, scalars, nullptr, skip, size, rowlen, table, N, c, J, nsets, st);
}
int grape_commit_fr_strided_masked_indexed(uint32_t* out, const uint32_t* entries, const int32_t* idx1, const int32_t* skip, size_t size, uint32_t rowlen,
                                           const uint32_t* table, size_t N, uint32_t c, uint32_t J, uint32_t nsets, grape_stream_t st) {
    GRAPE_REQUIRE(size == 0 || (skip != nullptr && idx1 != nullptr), "no flag or index array");
    return commit_strided_impl(out, entries, idx1, skip, size, rowlen, table, N, c, J, nsets, st);
}

int grape_g1_scaled_table_gen(uint32_t* out, const uint32_t* scalars, size_t len, size_t ncols, const uint32_t* table, size_t N,
                              uint32_t c, uint32_t nw, uint32_t K, grape_stream_t st) {
    CHECK_PTR16(out); CHECK_PTR16(scalars); CHECK_PTR16(table);
    GRAPE_REQUIRE(len >= 1 && ncols >= 1 && ncols <= N, "bad shape");
    GRAPE_REQUIRE(c >= 2 && c <= 16 && (uint64_t)nw * c >= 255 && K >= (1u << (c - 1)), "need a full-width wide table");
    hipStream_t s = as_stream(st);
    // slabs of scalars so that the XYZZ staging buffer stays near 1.5 GiB
    size_t slab = ((size_t)3 << 29) / (ncols * (16 * FW));
    if (slab < 1) slab = 1;
    if (slab > len) slab = len;
    void* ws;
    int rc = scratch_get(kSlotMsm, slab * ncols * (16 * FW) + 64, &ws, s);
    if (rc) return rc;
    int* err = (int*)((char*)ws + slab * ncols * (16 * FW));
    rc = zero_fill(err, sizeof(int), s);
    if (rc) return rc;
    for (size_t t0 = 0; t0 < len; t0 += slab) {
        size_t nt = len - t0 < slab ? len - t0 : slab;
        size_t n_entries = nt * ncols;
        scaled_chain_kernel<<<blocks_for(n_entries), kBlock, 0, s>>>((uint32_t*)ws, scalars, t0, nt, ncols, table, N, c, nw, K, err);
        size_t nthr = (n_entries + kNormChunk - 1) / kNormChunk;
        scaled_normalize_kernel<<<blocks_for(nthr, 64), 64, 0, s>>>(out, (const uint32_t*)ws, t0 * ncols, n_entries);
        GRAPE_LAUNCH_CHECK();
    }
    int h_err = 0;
    GRAPE_HIP_CHECK(hipMemcpyAsync(&h_err, err, sizeof(int), hipMemcpyDeviceToHost, s));
    GRAPE_HIP_CHECK(hipStreamSynchronize(s));
    if (h_err) {
        set_error("scaled table: a scalar digit exceeds the wide table's range");
        return GRAPE_EINVAL;
    }
    return GRAPE_OK;
}

static int commit_sparse_impl(uint32_t* out, const uint32_t* scalars, const int32_t* idx1, const int32_t* skip, size_t size, uint32_t rowlen,
                              const uint32_t* table, size_t N, uint32_t c, uint32_t nw, uint32_t K, grape_stream_t st) {
    if (size == 0) return GRAPE_OK;
    GRAPE_REQUIRE(size <= kMaxCommitScalars, "more than 2^28 scalars in one call: commit the rows in several calls");
    CHECK_PTR16(out); CHECK_PTR16(scalars); CHECK_PTR16(table);
    GRAPE_REQUIRE(skip != nullptr, "no flag array");
    GRAPE_REQUIRE(rowlen >= 1 && size % rowlen == 0, "size must be a multiple of rowlen");
    GRAPE_REQUIRE(rowlen <= N, "row longer than the generator set");
    GRAPE_REQUIRE(c >= 2 && c <= 16 && (uint64_t)nw * c >= 255 && K >= (1u << (c - 1)), "need a full-width wide table");
    const size_t rows = size / rowlen;
    hipStream_t s = as_stream(st);
    const size_t slab = rows < geom::kSlabSegments ? rows : geom::kSlabSegments;
    const size_t partial_bytes = slab * geom::kWaveLanes * (size_t)(4 * geom::kPartialWords);
    const size_t tmp_bytes = reduce_tmp_bytes(slab, geom::kWaveLanes);
    void* ws;
    int rc = scratch_get(kSlotMsm, partial_bytes + tmp_bytes + 64, &ws, s);
    if (rc) return rc;
    uint32_t* red_tmp = (uint32_t*)((char*)ws + partial_bytes);
    int* err = (int*)((char*)ws + partial_bytes + tmp_bytes);
    rc = zero_fill(err, sizeof(int), s);
    if (rc) return rc;
    for (size_t r0 = 0; r0 < rows; r0 += slab) {
        const size_t nr = rows - r0 < slab ? rows - r0 : slab;
        // many rows: half a wave per row, so that a thinly populated row still fills its batch
        const bool narrow = nr >= 4096;
        const uint32_t* sc = idx1 ? scalars : scalars + r0 * rowlen * 8;
        const int32_t* ix = idx1 ? idx1 + r0 * rowlen : nullptr;
        if (narrow)
            commit_sparse_fr_kernel<32><<<(unsigned)((nr + 1) / 2), 64, 0, s>>>((uint32_t*)ws, sc, ix, skip + r0 * rowlen, rowlen, nr,
                                                                              geom::spread_step((nr + 1) / 2), table, N, c, nw, K, err);
        else
            commit_sparse_fr_kernel<64><<<(unsigned)nr, 64, 0, s>>>((uint32_t*)ws, sc, ix, skip + r0 * rowlen, rowlen, nr,
                                                                   geom::spread_step(nr), table, N, c, nw, K, err);
        launch_reduce<true>(out + r0 * (size_t)(2 * FW), (const uint32_t*)ws, nr, narrow ? 32 : 64, red_tmp, s);
    }
    GRAPE_LAUNCH_CHECK();
    int h_err = 0;
    GRAPE_HIP_CHECK(hipMemcpyAsync(&h_err, err, sizeof(int), hipMemcpyDeviceToHost, s));
    GRAPE_HIP_CHECK(hipStreamSynchronize(s));
    if (h_err) {
        set_error("sparse commit: a scalar digit exceeds the wide table's range");
        return GRAPE_EINVAL;
    }
    return GRAPE_OK;
}

int grape_commit_fr_sparse(uint32_t* out, const uint32_t* scalars, const int32_t* skip, size_t size, uint32_t rowlen,
                           const uint32_t* table, size_t N, uint32_t c, uint32_t nw, uint32_t K, grape_stream_t st) {
    return commit_sparse_impl(out, scalars, nullptr, skip, size, rowlen, table, N, c, nw, K, st);
}
int grape_commit_fr_sparse_indexed(uint32_t* out, const uint32_t* entries, const int32_t* idx1, const int32_t* skip, size_t size, uint32_t rowlen,
                                   const uint32_t* table, size_t N, uint32_t c, uint32_t nw, uint32_t K, grape_stream_t st) {
    GRAPE_REQUIRE(size == 0 || idx1 != nullptr, "no index array");
    return commit_sparse_impl(out, entries, idx1, skip, size, rowlen, table, N, c, nw, K, st);
}

int grape_commit_i32(uint32_t* out, const int32_t* scalars, size_t size, uint32_t rowlen, const uint32_t* table, size_t N,
                     uint32_t c, uint32_t nw, uint32_t K, grape_stream_t st) {
    return commit_wide_impl<false>(out, scalars, size, rowlen, table, N, c, nw, K, st);
}
int grape_commit_i32_nowait(uint32_t* out, const int32_t* scalars, size_t size, uint32_t rowlen, const uint32_t* table, size_t N,
                            uint32_t c, uint32_t nw, uint32_t K, int32_t* d_flag, grape_stream_t st) {
    GRAPE_REQUIRE(d_flag != nullptr, "the caller's flag is required");
    return commit_wide_impl<false>(out, scalars, size, rowlen, table, N, c, nw, K, st, d_flag);
}
int grape_commit_start(uint32_t* out, const uint32_t* affine, grape_stream_t st) {
    CHECK_PTR16(out); CHECK_PTR16(affine);
    static_assert(GRAPE_COMMIT_START_WORDS == kPartialWords, "the header's accumulator is the kernels'");
    commit_start_kernel<<<1, 1, 0, as_stream(st)>>>(out, affine);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
int grape_commit_indexed(uint32_t* out, const int32_t* idx1, size_t size, uint32_t rowlen, const uint32_t* table, size_t ncols, uint32_t len, int32_t base1,
                         const uint32_t* start, int uneven, int32_t* d_flag, grape_stream_t st) {
    GRAPE_REQUIRE(len >= 1 && len <= (1u << 23), "between 1 and 2^23 entries");
    uint32_t c = 2;                                      // radix 2^c: a digit of up to 2^(c-1) with nothing above it stays positive
    while ((1u << (c - 1)) < len) c++;
    if (!start) return commit_wide_impl<false>(out, idx1, size, rowlen, table, ncols, c, 1, len, st, d_flag);
    CHECK_PTR16(start);
    const CommitBase base{start, base1, (size_t)(uneven ? 1 : 0)};
    return commit_wide_impl<false>(out, idx1, size, rowlen, table, ncols, c, 1, len, st, d_flag, &base);
}
int grape_commit_fr(uint32_t* out, const uint32_t* scalars, size_t size, uint32_t rowlen, const uint32_t* table, size_t N,
                    uint32_t c, uint32_t nw, uint32_t K, grape_stream_t st) {
    return commit_wide_impl<true>(out, scalars, size, rowlen, table, N, c, nw, K, st);
}
int grape_commit_fr_nowait(uint32_t* out, const uint32_t* scalars, size_t size, uint32_t rowlen, const uint32_t* table, size_t N,
                           uint32_t c, uint32_t nw, uint32_t K, int32_t* d_flag, grape_stream_t st) {
    GRAPE_REQUIRE(d_flag != nullptr, "the caller's flag is required");
    return commit_wide_impl<true>(out, scalars, size, rowlen, table, N, c, nw, K, st, d_flag);
}

int grape_commit_i32_ref_table(uint32_t* out, const int32_t* scalars, size_t size, uint32_t rowlen, const uint32_t* table,
                               size_t npoints, grape_stream_t st) {
    return commit_ref_impl<false>(out, scalars, size, rowlen, table, npoints, st);
}
int grape_commit_fr_ref_table(uint32_t* out, const uint32_t* scalars, size_t size, uint32_t rowlen, const uint32_t* table,
                              size_t npoints, grape_stream_t st) {
    return commit_ref_impl<true>(out, scalars, size, rowlen, table, npoints, st);
}

int grape_g1_msm_windows(uint32_t* sums, const uint32_t* points, const uint32_t* scalars, size_t n, grape_stream_t st) {
    GRAPE_REQUIRE(n >= 1 && n <= ((size_t)1 << 24), "between 1 and 2^24 points");
    CHECK_PTR16(sums); CHECK_PTR16(points); CHECK_PTR16(scalars);
    hipStream_t s = as_stream(st);
    // points go through in slabs, so that their multiples stay within 64 MiB
    const size_t slab = n < 32768 ? n : 32768;
    const size_t groups = (n + kMsmGroup - 1) / kMsmGroup;
    constexpr size_t kAcc = 4 * kPartialWords;
    const size_t table_bytes = slab * kMsmMultiples * kAcc, partial_bytes = groups * kMsmWindows * kAcc;
    void* ws;
    int rc = scratch_get(kSlotMsm, table_bytes + partial_bytes + reduce_tmp_bytes(kMsmWindows, (uint32_t)groups) + kMsmWindows * kAcc, &ws, s);
    if (rc) return rc;
    uint32_t* table = (uint32_t*)ws;
    uint32_t* partial = (uint32_t*)((char*)ws + table_bytes);
    uint32_t* total = (uint32_t*)((char*)partial + partial_bytes);
    uint32_t* tmp = (uint32_t*)((char*)total + kMsmWindows * kAcc);
    for (size_t i0 = 0; i0 < n; i0 += slab) {
        const size_t ni = n - i0 < slab ? n - i0 : slab;
        const uint32_t ng = (uint32_t)((ni + kMsmGroup - 1) / kMsmGroup);
        msm_multiples_kernel<<<blocks_for(ni * kMsmMultiples * 4), kBlock, 0, s>>>(table, points + 3 * FW * i0, ni);
        msm_window_kernel<<<blocks_for((size_t)kMsmWindows * ng * 64), kBlock, 0, s>>>(partial + (i0 / kMsmGroup) * kPartialWords, table, scalars + 8 * i0, ni, ng,
                                                                                   groups);
    }
    launch_reduce<false>(total, partial, kMsmWindows, (uint32_t)groups, tmp, s);
    quad_canonical_kernel<<<blocks_for(kMsmWindows * 4, 64), 64, 0, s>>>(sums, total, kMsmWindows);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

int grape_g1_affine_to_jacobian(uint32_t* out, const uint32_t* in, size_t n, grape_stream_t st) {
    if (n == 0) return GRAPE_OK;
    CHECK_PTR16(out); CHECK_PTR16(in);
    affine_to_jac_kernel<<<blocks_for(n, 64), 64, 0, as_stream(st)>>>(out, in, n);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
int grape_g1_jacobian_to_affine(uint32_t* out, const uint32_t* in, size_t n, grape_stream_t st) {
    if (n == 0) return GRAPE_OK;
    CHECK_PTR16(out); CHECK_PTR16(in);
    jac_to_affine_kernel<<<blocks_for(n, 64), 64, 0, as_stream(st)>>>(out, in, n);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

int grape_g1_affine_add(uint32_t* out, const uint32_t* a, const uint32_t* b, size_t n, grape_stream_t st) {
    if (n == 0) return GRAPE_OK;
    CHECK_PTR16(out); CHECK_PTR16(a); CHECK_PTR16(b);
    affine_add_kernel<<<blocks_for(n, 64), 64, 0, as_stream(st)>>>(out, a, b, n);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

}  // extern "C"
