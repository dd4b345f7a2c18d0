// Fr tensor kernels: element-wise field ops, integer embedding, Montgomery in/out, padding,
// reductions, batched inversion and the multilinear fold.
//
// Layout: a tensor is an array of 32-byte elements (the reference's fr_t array); every lane moves
// one element with two 16-byte vector accesses, so a wave64 covers 2 KiB of contiguous memory per
// element index and both halves of every 128-byte line are consumed back to back.
#include "fr_device.hpp"
#include <type_traits>
#include "divstep.hpp"

namespace grape {

// ------------------------------------------------------------------------------------------------
// element-wise
// ------------------------------------------------------------------------------------------------
enum BinOp { OP_ADD, OP_SUB, OP_MUL };

template <int OP>
__device__ __forceinline__ Fr apply(const Fr& a, const Fr& b) {
    if (OP == OP_ADD) return add(a, b);
    if (OP == OP_SUB) return sub(a, b);
    return fr26::mulc(a, b);
}

template <int OP>
__global__ void __launch_bounds__(kBlock) ew_kernel(uint32_t* out, const uint32_t* a, const uint32_t* b, size_t n) {
    size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    st_fr(out, i, apply<OP>(ld_fr(a, i), ld_fr(b, i)));
}

// plain copy with the tensors' access pattern (one 32-byte element per lane, two 16-byte accesses)
__global__ void __launch_bounds__(kBlock) copy_fr_kernel(uint32_t* out, const uint32_t* a, size_t n) {
    size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    st_fr(out, i, ld_fr(a, i));
}

template <int OP>
__global__ void __launch_bounds__(kBlock) bcast_kernel(uint32_t* out, const uint32_t* a, const uint32_t* x, size_t n) {
    size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    st_fr(out, i, apply<OP>(ld_fr(a, i), ld_fr(x, 0)));
}

// out = x + r * y with one scalar r (the combined witness of a mapping lookup, S_in + r * S_out,
// src/tlookup.cu:407-410, in one pass instead of a copy, a scalar product and a sum)
__global__ void __launch_bounds__(kBlock) axpy_kernel(uint32_t* out, const uint32_t* x, const uint32_t* r, const uint32_t* y, size_t n) {
    size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    st_fr(out, i, add(ld_fr(x, i), fr26::mulc(ld_fr(y, i), ld_fr(r, 0))));
}

__global__ void __launch_bounds__(kBlock) from_i32_kernel(uint32_t* out, const int32_t* in, size_t n) {
    size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    st_fr(out, i, fr26::from_i32c(in[i]));
}
__global__ void __launch_bounds__(kBlock) from_u32_kernel(uint32_t* out, const uint32_t* in, size_t n) {
    size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    st_fr(out, i, fr26::from_u32c(in[i]));
}
template <bool TO>
__global__ void __launch_bounds__(kBlock) mont_kernel(uint32_t* out, const uint32_t* in, size_t n) {
    size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    Fr a = ld_fr(in, i);
    st_fr(out, i, TO ? fr26::to_montc(a) : fr26::from_montc(a));
}

__global__ void __launch_bounds__(kBlock) pad_fr_kernel(uint32_t* out, const uint32_t* in, uint32_t N, uint32_t pad_N,
                                                        size_t size, const uint32_t* pad_val) {
    size_t g = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (g >= size) return;
    size_t row = g / pad_N;
    uint32_t col = (uint32_t)(g % pad_N);
    st_fr(out, g, col < N ? ld_fr(in, row * N + col) : ld_fr(pad_val, 0));
}
__global__ void __launch_bounds__(kBlock) pad_i32_kernel(int32_t* out, const int32_t* in, uint32_t N, uint32_t pad_N, size_t size,
                                                         int32_t fill) {
    size_t g = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (g >= size) return;
    size_t row = g / pad_N;
    uint32_t col = (uint32_t)(g % pad_N);
    out[g] = col < N ? in[row * N + col] : fill;
}

// ------------------------------------------------------------------------------------------------
// reductions
// ------------------------------------------------------------------------------------------------
// Grid-stride partial sums, one for each workgroup.  ONCE: the last workgroup to leave its own adds them up, so that a sum is
// one launch instead of two (*ticket is zero between launches).  Up to kSumOnce elements, over at most kSumOnceBlocks workgroups, behind
// a product of as many elements: 2^16 20.5 to 21.6 -> 18.2 to 18.9 us, 190 003 20.8 to 21.9 -> 18.3 to 19.3, 2^19 23.2 -> 20.8, most of it
// calls and launches (64 workgroups: 21.4 at 2^19, 256: 22.7).  From 2^20 elements on reading them is what takes the time: 32.5 us
// either way.  Every workgroup pays for a fence and for its turn at the counter, and where it is one of
// thousands that is more than a launch (2^20 elements 33 -> 52 us, 2^24 380 -> 473).
constexpr int kSumTerms = 4;               // loads a thread of a short sum has in flight
constexpr size_t kSumOnce = 1 << 19;
constexpr unsigned kSumOnceBlocks = 128;
template <bool ONCE>
__global__ void __launch_bounds__(kBlock) sum_kernel(uint32_t* out, const uint32_t* in, size_t n, uint32_t* partial, uint32_t* ticket) {
    __shared__ Fr lds[kBlock / 64];
    __shared__ uint32_t lds9[kBlock / 64 * 9], last;
    Fr acc = Fr::zero();
    const size_t stride = (size_t)gridDim.x * kBlock;
    size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    for (; ONCE && i + (kSumTerms - 1) * stride < n; i += kSumTerms * stride) {
        Fr x[kSumTerms];
#pragma unroll
        for (int k = 0; k < kSumTerms; k++) x[k] = ld_fr(in, i + k * stride);
#pragma unroll
        for (int k = 0; k < kSumTerms; k++) acc = add(acc, x[k]);
    }
    for (; i < n; i += stride) acc = add(acc, ld_fr(in, i));
    block_sum<1>(&acc, lds);
    if (!ONCE) {
        if (threadIdx.x == 0) st_fr(out, blockIdx.x, acc);
        return;
    }
    if (threadIdx.x == 0) {
        st_fr(partial, blockIdx.x, acc);
        __threadfence();
        last = atomicAdd(ticket, 1u) == gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    __threadfence();
    workgroup_totals<1, kBlock>(&acc, partial, gridDim.x, lds9);
    if (threadIdx.x == 0) {
        st_fr(out, 0, acc);
        *ticket = 0;
    }
}

__global__ void __launch_bounds__(kBlock) sum_by_dim_kernel(uint32_t* out, const uint32_t* in, size_t rows, size_t dim) {
    // one wave per row: strided partial sums, wave tree, broadcast back
    const int lane = threadIdx.x & 63;
    size_t row = ((size_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
    if (row >= rows) return;
    Fr acc = Fr::zero();
    for (size_t i = lane; i < dim; i += 64) acc = add(acc, ld_fr(in, row * dim + i));
    acc = wave_sum(acc);
    Fr tot;
#pragma unroll
    for (int k = 0; k < 8; k++) tot.v[k] = __shfl(acc.v[k], 0, 64);
    for (size_t i = lane; i < dim; i += 64) st_fr(out, row * dim + i, tot);
}

// ------------------------------------------------------------------------------------------------
// batched inversion (Montgomery's trick), three levels:
//   chunk products -> (recursive inversion of the products) -> back-substitution.
// Zero inputs are skipped in the products and produce zero outputs.
// ------------------------------------------------------------------------------------------------
constexpr int kInvChunk = 8;

// prod[t] = product of the non-zero elements of chunk t (beta added first when given)
__global__ void __launch_bounds__(kBlock) inv_prod_kernel(uint32_t* prod, const uint32_t* in, const uint32_t* beta, size_t n) {
    size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x;
    size_t nchunks = (n + kInvChunk - 1) / kInvChunk;
    if (t >= nchunks) return;
    Fr acc = Fr::one();
    Fr bt = beta ? ld_fr(beta, 0) : Fr::zero();
    // chunk t owns elements t, t + nchunks, t + 2*nchunks, ... so that lanes stay coalesced
#pragma unroll
    for (int k = 0; k < kInvChunk; k++) {
        size_t i = t + (size_t)k * nchunks;
        if (i < n) {
            Fr x = ld_fr(in, i);
            if (beta) x = add(x, bt);
            if (!x.is_zero()) acc = fr26::mulc(acc, x);
        }
    }
    st_fr(prod, t, acc);
}
// given inv_prod[t] = 1/prod[t], write the individual inverses.  Only the prefix products stay in
// registers (8 elements = 64 registers); the elements themselves are read again on the way back -
// holding both sets spilled to scratch memory, which cost 2.5 times the traffic of the second read.
__global__ void __launch_bounds__(kBlock) inv_back_kernel(uint32_t* out, const uint32_t* in, const uint32_t* beta,
                                                          const uint32_t* inv_prod, size_t n) {
    size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x;
    size_t nchunks = (n + kInvChunk - 1) / kInvChunk;
    if (t >= nchunks) return;
    Fr bt = beta ? ld_fr(beta, 0) : Fr::zero();
    Fr pre[kInvChunk];   // pre[k] = product of non-zero x[0..k-1]
    Fr acc = Fr::one();
#pragma clang loop unroll(full)
    for (int k = 0; k < kInvChunk; k++) {
        size_t i = t + (size_t)k * nchunks;
        Fr x = Fr::zero();
        if (i < n) {
            x = ld_fr(in, i);
            if (beta) x = add(x, bt);
        }
        pre[k] = acc;
        if (!x.is_zero()) acc = fr26::mulc(acc, x);
    }
    Fr inv = ld_fr(inv_prod, t);   // 1 / product of all non-zero x
#pragma clang loop unroll(full)
    for (int k = kInvChunk - 1; k >= 0; k--) {
        size_t i = t + (size_t)k * nchunks;
        if (i < n) {
            Fr x = ld_fr(in, i);          // (out may be in: element i is read before it is written, by this thread only)
            if (beta) x = add(x, bt);
            if (x.is_zero()) {
                st_fr(out, i, Fr::zero());
            } else {
                st_fr(out, i, fr26::mulc(inv, pre[k]));
                inv = fr26::mulc(inv, x);
            }
        }
    }
}
// direct inversion, used for the last (small) level
__global__ void __launch_bounds__(kBlock) inv_direct_kernel(uint32_t* out, const uint32_t* in, const uint32_t* beta, size_t n) {
    size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    Fr x = ld_fr(in, i);
    if (beta) x = add(x, ld_fr(beta, 0));
    st_fr(out, i, divstep::inverse_by(x));
}

// Uniformly random elements from a key: element i is the first of the 255-bit (BN254: 254-bit) numbers below the modulus in the ChaCha20
// key stream (RFC 8439) of the nonce (i, 0, 0), two candidates a block from block 0 on, read as memory form - what the host draws
// from the system's generator word by word.  A candidate is below r with probability 0.91 (BN254: 0.76): after 64 blocks, never in
// practice, the last one is reduced instead.  Bound by latency (a block is 80 dependent quarter rounds' depth): 4096 elements
// take 6 us where the host's draws took 160.
constexpr uint32_t kRandomBlocks = 64;
#if defined(GRAPE_CURVE_BN254)
constexpr int kRandomSpareBits = 2;        // r is a 254-bit number
#else
constexpr int kRandomSpareBits = 1;        // 255 bits
#endif
struct RandomKey { uint32_t w[8]; };
__device__ __forceinline__ void chacha_quarter(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d) {
    a += b; d = __builtin_rotateleft32(d ^ a, 16);
    c += d; b = __builtin_rotateleft32(b ^ c, 12);
    a += b; d = __builtin_rotateleft32(d ^ a, 8);
    c += d; b = __builtin_rotateleft32(b ^ c, 7);
}
__global__ void __launch_bounds__(64) random_kernel(uint32_t* out, size_t n, RandomKey key) {
    const size_t i = (size_t)blockIdx.x * 64 + threadIdx.x;
    if (i >= n) return;
    constexpr uint32_t kTop = 0xffffffffu >> kRandomSpareBits;
    Fr x = Fr::zero();
    bool found = false;
    for (uint32_t block = 0; block < kRandomBlocks && !found; block++) {
        const uint32_t init[16] = {0x61707865u, 0x3320646eu, 0x79622d32u, 0x6b206574u, key.w[0], key.w[1], key.w[2], key.w[3],
                                   key.w[4], key.w[5], key.w[6], key.w[7], block, (uint32_t)i, (uint32_t)((uint64_t)i >> 32), 0u};
        uint32_t s[16];
#pragma unroll
        for (int k = 0; k < 16; k++) s[k] = init[k];
        for (int round = 0; round < 10; round++) {
#pragma unroll
            for (int k = 0; k < 4; k++) chacha_quarter(s[k], s[4 + k], s[8 + k], s[12 + k]);
#pragma unroll
            for (int k = 0; k < 4; k++) chacha_quarter(s[k], s[4 + (k + 1) % 4], s[8 + (k + 2) % 4], s[12 + (k + 3) % 4]);
        }
#pragma unroll
        for (int half = 0; half < 2; half++) {
            if (found) break;
            uint32_t borrow = 0;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                x.v[k] = s[8 * half + k] + init[8 * half + k];
                if (k == 7) x.v[k] &= kTop;
                (void)detail::sbb32(x.v[k], FrParams::mod(k), borrow);
            }
            found = borrow != 0;
        }
    }
    if (!found) detail::final_sub<FrParams>(x.v, x.v, 0);
    st_fr(out, i, x);
}

// ------------------------------------------------------------------------------------------------
// fold.  One pass binds the TOP b bits of the folded axis (the multilinear extension does not
// care in which order variables are bound, and binding high bits keeps every access contiguous):
//   out[o][i_lo][g] = sum_{i_hi} w[i_hi] * t[o][i_hi*c_lo + i_lo][g],   i_hi*c_lo + i_lo < c
// with w[i_hi] = prod_k eq(x[k], bit_k(i_hi)) over the b challenges of those bits.
// ------------------------------------------------------------------------------------------------
constexpr int kFoldMaxBits = 8;      // bits bound by one pass (at most 64 products per thread)
constexpr int kFoldMaxPasses = 16;
constexpr int kFoldJobs = 2;         // tensors folded side by side (grape_fr_fold_pair): one launch serves a pass of both

struct FoldWeights {
    const uint32_t* x[kFoldJobs];
    uint32_t npass, npass0;                                     // passes of both, of the first
    uint32_t lo[kFoldJobs * kFoldMaxPasses];                    // the pass binds challenges lo .. lo+b-1
    uint32_t b[kFoldJobs * kFoldMaxPasses];
    uint32_t plain;                                             // bit p: pass p reads plain integers, its weights carry the factor 2^256 that
                                                                // brings a product with a plain value into memory form
};

// Weights of every pass of a fold, in the 26-bit working form with the radix factor 16 folded
// in (reduced mod r): workgroup p writes w[i] = prod_k eq(x[lo+k], bit_k(i)) for i < 2^b.
// Bound by the latency of dependent products: pairs of factors, then fours, then the weight - three products in a row, each on
// as many lanes as it has values (a tree of seven on every lane took 12 us for a fold, this 5).
__global__ void __launch_bounds__(kBlock) fold_weights_kernel(int32_t* wts, FoldWeights plan) {
    __shared__ Fr two[kFoldMaxBits / 2][4], four[2][16];
    const uint32_t p = blockIdx.x, b = plan.b[p], t = threadIdx.x;
    const uint32_t* x = plan.x[p >= plan.npass0];
    const bool plain = (plan.plain >> p) & 1;
    if (t < 2 * kFoldMaxBits) {
        const uint32_t k = 2 * (t >> 2);
        Fr f[2];
#pragma unroll
        for (uint32_t i = 0; i < 2; i++) {
            const Fr v = ld_fr(x, plan.lo[p] + (k + i < b ? k + i : 0));
            f[i] = k + i < b ? (((t >> i) & 1) ? v : sub(Fr::one(), v)) : Fr::one();
        }
        two[t >> 2][t & 3] = fr26::mulc(f[0], f[1]);
    }
    __syncthreads();
    if (t < 32) four[t >> 4][t & 15] = fr26::mulc(two[2 * (t >> 4)][t & 3], two[2 * (t >> 4) + 1][(t >> 2) & 3]);
    __syncthreads();
    if (t >= (1u << b)) return;
    Fr acc = four[0][t & 15];
    if (b > 4) acc = fr26::mulc(acc, four[1][t >> 4]);
    if (plain) acc = fr26::mulc(acc, Fr::rr());
    const fr26::Limbs w = fr26::weight16(acc);
    int32_t* dst = wts + (size_t)fr26::N * ((p << kFoldMaxBits) + t);
#pragma unroll
    for (int k = 0; k < fr26::N; k++) dst[k] = w.v[k];
}

// one tensor's part of a pass
struct FoldJob {
    uint32_t* out;
    const uint32_t* in;
    const int32_t* wts;
    uint32_t n_hi_max, outer, c, lg_c_lo, gap;
};
struct FoldPassArgs {
    FoldJob job[kFoldJobs];
    uint32_t blocks0;                  // the first tensor's workgroups; the others are the second's
};

// an integer x = l0 + 2^26 l1 with 0 <= l0 < 2^26, -32 <= l1 < 32: a column grows by < 2^53 per term
__device__ __forceinline__ void fold_mac_int(fr26::Acc& C, const fr26::Limbs& w, int32_t xv) {
    const int64_t l0 = (int64_t)(xv & (int32_t)fr26::MASK), l1 = (int64_t)(xv >> fr26::W);
#pragma unroll
    for (int j = 0; j < fr26::N; j++) {
        C.c[j] += (int64_t)w.v[j] * l0;
        C.c[j + 1] += (int64_t)w.v[j] * l1;
    }
}

// One pass.  A workgroup is 4 waves: 4/S groups of 64 outputs, each output summed by S waves
// that take every S-th term; the partial sums meet in LDS.  The weight index is wave-uniform, so
// the weights arrive through scalar loads and cost no vector registers.
// I32: the input is a tensor of 32-bit integers (the value x stands for the field element x, negative values for
// r - |x|): an element is two signed limbs, a product 20 multiply-adds, and 4 bytes are read where the embedded
// tensor has 32 - the pass that folds an integer tensor without first writing it out as field elements.
template <int S, bool I32 = false>
__global__ void __launch_bounds__(kBlock) fold_pass_kernel(FoldPassArgs args) {
    constexpr int IW = 4 / S;                       // output groups per workgroup
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int iw = wave % IW, part = wave / IW;
    const bool second = blockIdx.x >= args.blocks0;
    const FoldJob& job = args.job[second];
    uint32_t* __restrict__ out = job.out;
    const uint32_t* __restrict__ in = job.in;
    const int32_t* __restrict__ wts = job.wts;
    const uint32_t c = job.c, lg_c_lo = job.lg_c_lo, gap = job.gap, n_hi_max = job.n_hi_max;
    // index arithmetic in 32 bits (the host checks that the output count fits)
    const uint32_t c_lo = 1u << lg_c_lo;
    const uint32_t c_out = c < c_lo ? c : c_lo;     // surviving extent of the axis
    const uint32_t inner = c_out * gap;             // outputs per outer index
    const uint32_t total = job.outer * inner;
    const uint32_t tid = (((uint32_t)blockIdx.x - (second ? args.blocks0 : 0u)) * IW + iw) * 64 + lane;
    const bool live = tid < total;
    const uint32_t o = live ? tid / inner : 0;
    const uint32_t p = live ? tid - o * inner : 0;  // i_lo*gap + g
    const uint32_t i_lo = p / gap;
    const uint32_t* src = in + (I32 ? 1 : 8) * ((size_t)o * c * gap + p);
    const int32_t* isrc = reinterpret_cast<const int32_t*>(src);
    const size_t hi_stride = (size_t)c_lo * gap;    // elements between consecutive i_hi
    // number of i_hi with i_hi*c_lo + i_lo < c (zero for a dead lane)
    const uint32_t n_hi = live ? (c - i_lo + c_lo - 1) >> lg_c_lo : 0;
    // One double-width accumulator per thread: at most 64 products of values below r, so the
    // column sums stay below 64 * 10 * 2^52 and the reduced value below 2.82 r.
    fr26::Acc C;
    fr26::acc_zero(C);
    // Terms below n_full = c / c_lo exist for every lane, so the main loop is branch-free with
    // wave-uniform offsets and four loads in flight per lane (a dead lane reads the terms of
    // output 0 and stores nothing).  A ragged last term (c not a multiple of c_lo) follows
    // under a lane predicate, in the part whose turn it is.
    constexpr int U = I32 ? 8 : 4;
    const uint32_t n_full = c >> lg_c_lo;
    uint32_t h = (uint32_t)part;
    for (; h + (U - 1) * S < n_full; h += U * S) {
        Fr t[I32 ? 1 : U];
        int32_t ti[I32 ? U : 1];
#pragma unroll
        for (int k = 0; k < U; k++) {
            if (I32) ti[k] = isrc[(size_t)(h + k * S) * hi_stride];
            else t[k] = ld_fr(src, (size_t)(h + k * S) * hi_stride);
        }
#pragma unroll
        for (int k = 0; k < U; k++) {
            fr26::Limbs w;
#pragma unroll
            for (int j = 0; j < fr26::N; j++) w.v[j] = wts[(size_t)fr26::N * (h + k * S) + j];
            if (I32) fold_mac_int(C, w, ti[k]);
            else fr26::mac(C, w, fr26::pack(t[k]));
        }
    }
    for (; h < n_hi_max; h += S) {
        if (h < n_hi) {
            fr26::Limbs w;
#pragma unroll
            for (int j = 0; j < fr26::N; j++) w.v[j] = wts[(size_t)fr26::N * h + j];
            if (I32) fold_mac_int(C, w, isrc[(size_t)h * hi_stride]);
            else fr26::mac(C, w, ld_l26(src, (size_t)h * hi_stride));
        }
    }
    fr26::Limbs r = fr26::reduce(C, 0);
    if (S > 1) {
        __shared__ int32_t lds[fr26::N * (S > 1 ? S - 1 : 1) * IW * 64];
        if (part > 0) {
#pragma unroll
            for (int k = 0; k < fr26::N; k++) lds[((k * (S - 1) + part - 1) * IW + iw) * 64 + lane] = r.v[k];
        }
        __syncthreads();
        if (part == 0) {
#pragma unroll
            for (int q = 1; q < S; q++) {
#pragma unroll
                for (int k = 0; k < fr26::N; k++) r.v[k] += lds[((k * (S - 1) + q - 1) * IW + iw) * 64 + lane];
            }
            r = fr26::normalize(r);
        }
    }
    // below 2.82 S r <= 11.3 r
    if (part == 0 && live) st_fr(out, tid, fr26::unpack(fr26::canon_wide(r)));
}

// A pass with few outputs: 256 / P of them a workgroup, each summed by P of its threads, P = 16 or 256, so that a chain of
// terms is a sixteenth as long and the outputs of a short pass still fill the chip.  Two operands' 4096 outputs of 128 terms: 11 us
// where four waves an output took 2 x 8 for 8 terms each and left the rest to a workgroup per outer index (2 x 13).  P threads' sums of at most 256 / P
// products each: P = 16, 16 (1 + 16 / 35.3) r = 23.3 r at most; P = 256, 16 (1 + 1 / 35.3) r = 16.5 r in a row of lanes.
template <int P, bool I32 = false>
__global__ void __launch_bounds__(kBlock) fold_short_kernel(FoldPassArgs args) {
    static_assert(P == 16 || P == 256, "parts that meet in LDS resp. in a row of lanes first");
    constexpr int OW = kBlock / P;
    const bool second = blockIdx.x >= args.blocks0;
    const FoldJob& job = args.job[second];
    const uint32_t c = job.c, lg_c_lo = job.lg_c_lo, gap = job.gap;
    const uint32_t c_lo = 1u << lg_c_lo, c_out = c < c_lo ? c : c_lo, inner = c_out * gap, total = job.outer * inner;
    const uint32_t o_in = threadIdx.x % OW, part = threadIdx.x / OW;
    const uint32_t q = ((uint32_t)blockIdx.x - (second ? args.blocks0 : 0u)) * OW + o_in;
    const bool live = q < total;
    const uint32_t o = live ? q / inner : 0, p = live ? q - o * inner : 0, i_lo = p / gap;
    const size_t first = (size_t)o * c * gap + p, hi_stride = (size_t)c_lo * gap;
    const uint32_t n_hi = live ? (c - i_lo + c_lo - 1) >> lg_c_lo : 0;
    const int32_t* in32 = reinterpret_cast<const int32_t*>(job.in);
    fr26::Acc C;
    fr26::acc_zero(C);
    auto terms = [&](uint32_t h, auto count) {      // `count` terms, all their operands asked for before the first is used
        constexpr int U = decltype(count)::value;
        Fr t[U];
        int32_t ti[U];
        fr26::Limbs w[U];
#pragma unroll
        for (int k = 0; k < U; k++) {
            if (I32) ti[k] = in32[first + (h + k * P) * hi_stride];
            else t[k] = ld_fr(job.in, first + (h + k * P) * hi_stride);
            const int2* wp = reinterpret_cast<const int2*>(job.wts + (size_t)fr26::N * (h + k * P));
#pragma unroll
            for (int j = 0; j < fr26::N / 2; j++) {
                const int2 v = wp[j];
                w[k].v[2 * j] = v.x;
                w[k].v[2 * j + 1] = v.y;
            }
        }
        __builtin_amdgcn_sched_barrier(0);          // the compiler would ask for each where it is used: a round trip a term
#pragma unroll
        for (int k = 0; k < U; k++) {
            if (I32) fold_mac_int(C, w[k], ti[k]);
            else fr26::mac(C, w[k], fr26::pack(t[k]));
        }
    };
    uint32_t h = part;
    if (P == 16)
        for (; h + 3 * P < n_hi; h += 4 * P) terms(h, std::integral_constant<int, 4>());
    for (; h < n_hi; h += P) terms(h, std::integral_constant<int, 1>());
    fr26::Limbs r = fr26::reduce(C, 0);
    if constexpr (P == 16) {
        __shared__ int32_t lds[fr26::N][kBlock + OW];
#pragma unroll
        for (int k = 0; k < fr26::N; k++) lds[k][threadIdx.x] = r.v[k];
        __syncthreads();
        if (threadIdx.x < fr26::N * OW) {
            const uint32_t k = threadIdx.x / OW, oo = threadIdx.x % OW;
            int32_t sum = 0;
#pragma unroll
            for (int i = 0; i < P; i++) sum += lds[k][i * OW + oo];
            lds[k][kBlock + oo] = sum;
        }
        __syncthreads();
        if (part == 0 && live) {
#pragma unroll
            for (int k = 0; k < fr26::N; k++) r.v[k] = lds[k][kBlock + o_in];
            st_fr(job.out, q, fr26::unpack(fr26::canon_wide(fr26::normalize(r))));
        }
    } else {
        __shared__ Fr rows[kBlock / 16];
        const Fr f = fr26::limb_sum_to_fr(row_sum(r), 0);
        if ((threadIdx.x & 15) == 15) rows[threadIdx.x >> 4] = f;
        __syncthreads();
        if (threadIdx.x < 64) {
            const Fr s = fr26::limb_sum_to_fr(row_sum(fr26::pack(rows[threadIdx.x & 15])), 0);
            if (threadIdx.x == 15 && live) st_fr(job.out, q, s);
        }
    }
}

static uint32_t log2ceil(size_t n) {
    uint32_t r = 0;
    while (((size_t)1 << r) < n) r++;
    return r;
}

// Small-tensor finish: one workgroup holds the whole [c][gap] slab of one outer index in LDS
// and binds the remaining bits top-down with a barrier per level.
constexpr int kFoldSmallElems = 2048;   // 64 KiB of LDS
constexpr int kFoldSmallMaxOuter = 256; // one workgroup per outer index: worth it only for few
// Only the whole of a fold that is short anyway, which needs no weights then.  A workgroup's time is 0.9 us a step of 256 outputs; in
// steps (one call after another, launches included): one slab 16 x 16 4 steps 7.7 us, 32 x 16 5 7.7, 64 x 16 7 9.6, 256 8 10.6, 512 9 12.0,
// 32 x 64 9 11.6, 1024 11 14.1, 2048 15 18.4, where a pass takes 11.0 and two of them, for more than eight variables, 13.8; 16 slabs
// of 64 x 16 7 11.8, of 512 9 14.8, of 128 x 16 11 16.1 against 13.7.  Two folds side by side share their passes'
// launches and keep to slabs of an element a thread, or two variables, as do integers, which would be embedded first.
static bool fold_small_fits(size_t outer, size_t c, size_t gap, bool alone) {
    if (c * gap > (size_t)kFoldSmallElems || outer > (size_t)kFoldSmallMaxOuter) return false;
    if (!alone) return c <= 4 || c * gap <= (size_t)kBlock;
    const uint32_t L = log2ceil((uint32_t)c);
    size_t steps = 0;
    for (uint32_t l = 0; l < L; l++) steps += (gap << l) / kBlock + ((gap << l) % kBlock != 0);
    return steps <= (outer == 1 && L > (uint32_t)kFoldMaxBits ? 9u : 8u);
}

__global__ void __launch_bounds__(kBlock) fold_small_kernel(uint32_t* out, const uint32_t* in, const uint32_t* x,
                                                            uint32_t L, size_t c, size_t gap) {
    __shared__ Fr buf[kFoldSmallElems];
    const size_t o = blockIdx.x;
    const size_t n = c * gap;
    for (size_t i = threadIdx.x; i < n; i += kBlock) buf[i] = ld_fr(in, o * n + i);
    __syncthreads();
    size_t cur = c;
    for (int lvl = (int)L - 1; lvl >= 0; lvl--) {
        const size_t half = (size_t)1 << lvl;        // axis indices >= half fold onto [0, half)
        if (cur > half) {
            const Fr xv = ld_fr(x, lvl);
            const size_t nlow = half * gap;
            for (size_t i = threadIdx.x; i < nlow; i += kBlock) {
                const size_t j = i + nlow;
                Fr lo = buf[i];
                Fr hi = (j < cur * gap) ? buf[j] : Fr::zero();
                buf[i] = add(lo, fr26::mulc(xv, sub(hi, lo)));
            }
            cur = half;
        } else {
            // the whole upper half is padding: value *= (1 - x)
            const Fr xv = sub(Fr::one(), ld_fr(x, lvl));
            for (size_t i = threadIdx.x; i < cur * gap; i += kBlock) buf[i] = fr26::mulc(buf[i], xv);
        }
        __syncthreads();
    }
    for (size_t i = threadIdx.x; i < gap; i += kBlock) st_fr(out, o * gap + i, buf[i]);
}

}  // namespace grape

using namespace grape;


template <int OP>
static int launch_ew(uint32_t* out, const uint32_t* a, const uint32_t* b, size_t n, grape_stream_t st) {
    if (n == 0) return GRAPE_OK;
    CHECK_PTR16(out); CHECK_PTR16(a); CHECK_PTR16(b);
    ew_kernel<OP><<<blocks_for(n), kBlock, 0, as_stream(st)>>>(out, a, b, n);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
template <int OP>
static int launch_bcast(uint32_t* out, const uint32_t* a, const uint32_t* x, size_t n, grape_stream_t st) {
    if (n == 0) return GRAPE_OK;
    CHECK_PTR16(out); CHECK_PTR16(a); CHECK_PTR16(x);
    bcast_kernel<OP><<<blocks_for(n), kBlock, 0, as_stream(st)>>>(out, a, x, n);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

// shared by grape_fr_batch_inverse / grape_fr_shift_inverse
static int batch_inverse_impl(uint32_t* out, const uint32_t* in, const uint32_t* beta, size_t n, hipStream_t s) {
    if (n == 0) return GRAPE_OK;
    if (n <= 4096) {
        inv_direct_kernel<<<blocks_for(n), kBlock, 0, s>>>(out, in, beta, n);
        GRAPE_LAUNCH_CHECK();
        return GRAPE_OK;
    }
    // levels of chunk products live back to back in one scratch buffer
    size_t sizes[16];
    int levels = 0;
    size_t cur = n, total = 0;
    while (cur > 4096) {
        cur = (cur + kInvChunk - 1) / kInvChunk;
        sizes[levels++] = cur;
        total += cur;
    }
    void* ws;
    int rc = scratch_get(kSlotInv, total * 32, &ws, s);
    if (rc) return rc;
    uint32_t* lvl[16];
    {
        uint32_t* p = (uint32_t*)ws;
        for (int l = 0; l < levels; l++) {
            lvl[l] = p;
            p += 8 * sizes[l];
        }
    }
    // forward: products
    inv_prod_kernel<<<blocks_for(sizes[0]), kBlock, 0, s>>>(lvl[0], in, beta, n);
    for (int l = 1; l < levels; l++)
        inv_prod_kernel<<<blocks_for(sizes[l]), kBlock, 0, s>>>(lvl[l], lvl[l - 1], nullptr, sizes[l - 1]);
    // top: direct inversion in place
    inv_direct_kernel<<<blocks_for(sizes[levels - 1]), kBlock, 0, s>>>(lvl[levels - 1], lvl[levels - 1], nullptr, sizes[levels - 1]);
    // backward: each level's inverses from the level above (in place over the products)
    for (int l = levels - 1; l >= 1; l--)
        inv_back_kernel<<<blocks_for(sizes[l]), kBlock, 0, s>>>(lvl[l - 1], lvl[l - 1], nullptr, lvl[l], sizes[l - 1]);
    inv_back_kernel<<<blocks_for(sizes[0]), kBlock, 0, s>>>(out, in, beta, lvl[0], n);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

extern "C" {

int grape_fr_add(uint32_t* o, const uint32_t* a, const uint32_t* b, size_t n, grape_stream_t s) { return launch_ew<OP_ADD>(o, a, b, n, s); }
int grape_fr_sub(uint32_t* o, const uint32_t* a, const uint32_t* b, size_t n, grape_stream_t s) { return launch_ew<OP_SUB>(o, a, b, n, s); }
int grape_fr_mul(uint32_t* o, const uint32_t* a, const uint32_t* b, size_t n, grape_stream_t s) { return launch_ew<OP_MUL>(o, a, b, n, s); }
int grape_fr_bcast_add(uint32_t* o, const uint32_t* a, const uint32_t* x, size_t n, grape_stream_t s) { return launch_bcast<OP_ADD>(o, a, x, n, s); }
int grape_fr_bcast_mul(uint32_t* o, const uint32_t* a, const uint32_t* x, size_t n, grape_stream_t s) { return launch_bcast<OP_MUL>(o, a, x, n, s); }

int grape_bench_copy_fr(uint32_t* out, const uint32_t* in, size_t n, int iters, float* ms, grape_stream_t st) {
    CHECK_PTR16(out); CHECK_PTR16(in);
    GRAPE_REQUIRE(n > 0 && iters > 0 && ms != nullptr, "bad arguments");
    hipStream_t s = as_stream(st);
    hipEvent_t e0, e1;
    GRAPE_HIP_CHECK(hipEventCreate(&e0));
    GRAPE_HIP_CHECK(hipEventCreate(&e1));
    copy_fr_kernel<<<blocks_for(n), kBlock, 0, s>>>(out, in, n);
    GRAPE_HIP_CHECK(hipEventRecord(e0, s));
    for (int i = 0; i < iters; i++) copy_fr_kernel<<<blocks_for(n), kBlock, 0, s>>>(out, in, n);
    GRAPE_HIP_CHECK(hipEventRecord(e1, s));
    GRAPE_HIP_CHECK(hipEventSynchronize(e1));
    GRAPE_LAUNCH_CHECK();
    float t;
    GRAPE_HIP_CHECK(hipEventElapsedTime(&t, e0, e1));
    *ms = t / iters;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return GRAPE_OK;
}

int grape_fr_axpy(uint32_t* out, const uint32_t* x, const uint32_t* r, const uint32_t* y, size_t n, grape_stream_t st) {
    if (n == 0) return GRAPE_OK;
    CHECK_PTR16(out); CHECK_PTR16(x); CHECK_PTR16(r); CHECK_PTR16(y);
    axpy_kernel<<<blocks_for(n), kBlock, 0, as_stream(st)>>>(out, x, r, y, n);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
int grape_fr_from_i32(uint32_t* out, const int32_t* in, size_t n, grape_stream_t st) {
    if (n == 0) return GRAPE_OK;
    CHECK_PTR16(out);
    GRAPE_REQUIRE(in != nullptr, "null input");
    from_i32_kernel<<<blocks_for(n), kBlock, 0, as_stream(st)>>>(out, in, n);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
int grape_fr_from_u32(uint32_t* out, const uint32_t* in, size_t n, grape_stream_t st) {
    if (n == 0) return GRAPE_OK;
    CHECK_PTR16(out);
    GRAPE_REQUIRE(in != nullptr, "null input");
    from_u32_kernel<<<blocks_for(n), kBlock, 0, as_stream(st)>>>(out, in, n);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
int grape_fr_to_mont(uint32_t* out, const uint32_t* in, size_t n, grape_stream_t st) {
    if (n == 0) return GRAPE_OK;
    CHECK_PTR16(out); CHECK_PTR16(in);
    mont_kernel<true><<<blocks_for(n), kBlock, 0, as_stream(st)>>>(out, in, n);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
int grape_fr_from_mont(uint32_t* out, const uint32_t* in, size_t n, grape_stream_t st) {
    if (n == 0) return GRAPE_OK;
    CHECK_PTR16(out); CHECK_PTR16(in);
    mont_kernel<false><<<blocks_for(n), kBlock, 0, as_stream(st)>>>(out, in, n);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
int grape_fr_batch_inverse(uint32_t* out, const uint32_t* in, size_t n, grape_stream_t st) {
    if (n == 0) return GRAPE_OK;
    CHECK_PTR16(out); CHECK_PTR16(in);
    return batch_inverse_impl(out, in, nullptr, n, as_stream(st));
}
int grape_fr_shift_inverse(uint32_t* out, const uint32_t* in, const uint32_t* beta, size_t n, grape_stream_t st) {
    if (n == 0) return GRAPE_OK;
    CHECK_PTR16(out); CHECK_PTR16(in); CHECK_PTR16(beta);
    return batch_inverse_impl(out, in, beta, n, as_stream(st));
}

int grape_fr_sum(uint32_t* out, const uint32_t* in, size_t n, grape_stream_t st) {
    CHECK_PTR16(out);
    hipStream_t s = as_stream(st);
    if (n == 0) {
        return zero_fill(out, 32, s);
    }
    CHECK_PTR16(in);
    if (n <= kBlock * kSumTerms) {
        sum_kernel<false><<<1, kBlock, 0, s>>>(out, in, n, nullptr, nullptr);
        GRAPE_LAUNCH_CHECK();
        return GRAPE_OK;
    }
    const bool once = n <= kSumOnce;
    unsigned nb = blocks_for(n, once ? kBlock * kSumTerms : kBlock);
    const unsigned most = once ? kSumOnceBlocks : kNumCU * 8;
    if (nb > most) nb = most;
    void *ws, *ticket;
    int rc = scratch_get(kSlotReduce, (size_t)nb * 32, &ws, s);
    if (rc) return rc;
    if (once) {
        if ((rc = scratch_get(kSlotTicket, sizeof(uint32_t), &ticket, s))) return rc;
        sum_kernel<true><<<nb, kBlock, 0, s>>>(out, in, n, (uint32_t*)ws, (uint32_t*)ticket);
    } else {
        sum_kernel<false><<<nb, kBlock, 0, s>>>((uint32_t*)ws, in, n, nullptr, nullptr);
        launch_final_sum<1>(out, (const uint32_t*)ws, nb, s);
    }
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

int grape_fr_sum_by_dim(uint32_t* out, const uint32_t* in, size_t rows, size_t dim, grape_stream_t st) {
    if (rows == 0 || dim == 0) return GRAPE_OK;
    CHECK_PTR16(out); CHECK_PTR16(in);
    sum_by_dim_kernel<<<blocks_for(rows * 64), kBlock, 0, as_stream(st)>>>(out, in, rows, dim);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

int grape_fr_pad(uint32_t* out, const uint32_t* in, uint32_t N, uint32_t pad_N, size_t pad_size, const uint32_t* pad_val, grape_stream_t st) {
    if (pad_size == 0) return GRAPE_OK;
    CHECK_PTR16(out); CHECK_PTR16(in); CHECK_PTR16(pad_val);
    GRAPE_REQUIRE(N <= pad_N && pad_N > 0 && out != in, "need N <= pad_N and distinct buffers");
    pad_fr_kernel<<<blocks_for(pad_size), kBlock, 0, as_stream(st)>>>(out, in, N, pad_N, pad_size, pad_val);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
int grape_i32_pad(int32_t* out, const int32_t* in, uint32_t N, uint32_t pad_N, size_t pad_size, grape_stream_t st) {
    if (pad_size == 0) return GRAPE_OK;
    GRAPE_REQUIRE(out && in && N <= pad_N && pad_N > 0 && out != in, "need N <= pad_N and distinct buffers");
    pad_i32_kernel<<<blocks_for(pad_size), kBlock, 0, as_stream(st)>>>(out, in, N, pad_N, pad_size, 0);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}
int grape_i32_pad_fill(int32_t* out, const int32_t* in, uint32_t N, uint32_t pad_N, size_t pad_size, int32_t fill, grape_stream_t st) {
    if (pad_size == 0) return GRAPE_OK;
    GRAPE_REQUIRE(out && in && N <= pad_N && pad_N > 0 && out != in, "need N <= pad_N and distinct buffers");
    pad_i32_kernel<<<blocks_for(pad_size), kBlock, 0, as_stream(st)>>>(out, in, N, pad_N, pad_size, fill);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

// Plan of a fold's passes.  While a pass has outputs enough to fill the chip it binds as many top bits as it can stream; behind those
// the passes are short, bound by the chain of terms of one output, and bind up to eight bits each.
struct FoldPass { uint32_t b, P; };                // bits, parts that share an output
struct FoldPlan {
    uint32_t npass;
    FoldPass pass[kFoldMaxPasses];
    uint32_t lo[kFoldMaxPasses];
};
// Parts per output of a short pass over n_out outputs and 2^b terms: 125 instructions a term, 350 for the reduction of a part's sum
// and what the parts take to meet; a lone wave on a SIMD issues one instruction every 6.5 cycles, more of them one every 4.4.
static uint32_t short_pass_parts(size_t n_out, uint32_t b) {
    uint32_t best = 0;
    double best_t = 0;
    for (uint32_t P : {1u, 2u, 4u, 16u, 256u}) {
        if (P < 4 && (1u << b) > 64 * P) continue;
        const uint32_t terms = ((1u << b) + P - 1) / P;
        const double meet = P == 1 ? 0 : P < 16 ? 80 : P == 16 ? 150 : 300;
        const double waves = (double)n_out * P / (64 * 4 * kNumCU);
        const double t = (125.0 * terms + 350 + meet) * (4.4 * waves > 6.5 ? 4.4 * waves : 6.5);
        if (best == 0 || t < best_t) {
            best = P;
            best_t = t;
        }
    }
    return best;
}
static int plan_fold(size_t outer, uint32_t c, uint32_t gap, uint32_t id, bool ints, bool alone, FoldPlan& plan) {
    plan.npass = 0;
    uint32_t l = log2ceil(c);
    if (fold_small_fits(outer, c, gap, alone && !ints)) return GRAPE_OK;
    while (l > 0) {
        // Measured on MI355X: a pass streams fastest with one thread per output, 16 to 64
        // terms per thread and 2^20 threads; 2^19 threads come close.  Failing that, up to
        // four waves share an output to reach 2^19 threads.  A pass over integers reads an eighth of the bytes and is bound by
        // instructions, of which a thread's reduction is as many as 16 terms: 2^17 threads of up to 64 terms there (2048 x 4096
        // integers 30 -> 24 us, 4096 x 4096 45 -> 32, 2048 x 11008 53 -> 39, no size slower; 16 loads in flight instead of 8: no faster).
        const bool plain = ints && plan.npass == 0;
        const uint32_t most = plain ? 17 : 20, least = plain ? 17 : 19;
        uint32_t P = 0, b = 0;
        auto items = [&](uint32_t tb) { return outer * gap * ((size_t)1 << (l - tb)); };
        for (uint32_t want = most; want >= least && P == 0; want--) {
            for (uint32_t tb = l < 6 ? l : 6; tb >= 4 && P == 0; tb--) {
                if (items(tb) >= ((size_t)1 << want)) { P = 1; b = tb; }
            }
        }
        for (uint32_t tb = l < 8 ? l : 8; tb >= 4 && P == 0; tb--) {
            const uint32_t ts = items(tb) * 2 >= ((size_t)1 << 19) ? 2 : 4;
            if (items(tb) * ts >= ((size_t)1 << 19) && (1u << tb) <= 64 * ts) { P = ts; b = tb; }
        }
        if (P == 0) {
            // too few outputs to fill the chip whatever the split: as few passes as there can be, of about the same length
            const uint32_t left = (l + kFoldMaxBits - 1) / kFoldMaxBits;
            b = (l + left - 1) / left;
            P = short_pass_parts(items(b), b);
        }
        GRAPE_REQUIRE(plan.npass < (uint32_t)kFoldMaxPasses, "fold: too many passes");
        plan.pass[plan.npass] = {b, P};
        plan.lo[plan.npass] = id + (l - b);
        plan.npass++;
        l -= b;
    }
    return GRAPE_OK;
}

// The fold of one tensor on its way through its passes.
// With a single outer index a pass can run in place (an output's threads read nothing that another output is left in).
// Otherwise passes ping-pong through scratch and the last one writes to the front.
struct FoldRun {
    const grape_fold_job* j;
    FoldPlan plan;
    size_t outer, cur_c;
    uint32_t L, pi;
    bool ints, done;
    const uint32_t* src;
    size_t each;                       // elements of one scratch buffer, 0: none
    uint32_t* ws[2];
    int which;
    const int32_t* wts;
};
static int fold_start(FoldRun& r, const grape_fold_job& j, bool alone, hipStream_t s) {
    r = FoldRun{};
    r.j = &j;
    r.done = j.N == 0;
    if (r.done) return GRAPE_OK;
    CHECK_PTR16(j.t); CHECK_PTR16(j.x);
    GRAPE_REQUIRE(j.c >= 1 && j.gap >= 1 && j.N >= (size_t)j.c * j.gap && j.N % ((size_t)j.c * j.gap) == 0, "N must be a multiple of c*gap");
    GRAPE_REQUIRE(!j.from || !j.ints, "one source");
    if (j.from) {
        CHECK_PTR16(j.from);
        GRAPE_REQUIRE(j.from != j.t, "the source is kept: grape_fr_fold folds in place");
    }
    r.outer = j.N / ((size_t)j.c * j.gap);
    r.cur_c = j.c;
    r.L = log2ceil(j.c);
    int rc = plan_fold(r.outer, j.c, j.gap, j.id, j.ints != nullptr, alone, r.plan);
    if (rc) return rc;
    r.ints = j.ints != nullptr;
    if (r.ints && (r.L == 0 || r.plan.npass == 0)) {
        // nothing to bind, or a tensor small enough for the finish kernel alone: embedded first (N elements of t)
        from_i32_kernel<<<blocks_for(j.N), kBlock, 0, s>>>(j.t, j.ints, j.N);
        GRAPE_LAUNCH_CHECK();
        r.ints = false;
    }
    r.src = r.ints ? reinterpret_cast<const uint32_t*>(j.ints) : j.from ? j.from : j.t;
    if (r.L == 0) {                // c == 1: nothing to bind, data already compact
        if (j.from) GRAPE_HIP_CHECK(hipMemcpyAsync(j.t, j.from, j.N * 32, hipMemcpyDeviceToDevice, s));
        r.done = true;
        return GRAPE_OK;
    }
    // a single pass from another tensor writes to the front; with several outer indices the others go through scratch, the largest first
    if (r.outer > 1) {
        const uint32_t first = r.plan.npass ? r.L - r.plan.pass[0].b : 0;
        const size_t c_out = r.cur_c < ((size_t)1 << first) ? r.cur_c : (size_t)1 << first;
        if (r.plan.npass > 1 || r.src == j.t) r.each = r.outer * c_out * j.gap;
    }
    return GRAPE_OK;
}
// where the next pass, which leaves `c_out` of the axis, writes
static uint32_t* fold_target(FoldRun& r, bool last) {
    if (r.outer == 1 || (last && r.src != r.j->t)) return r.j->t;
    uint32_t* dst = r.ws[r.which];
    r.which ^= 1;
    return dst;
}
static int fold_next(FoldRun& r, FoldJob& out, uint32_t& total) {
    const FoldPass& ps = r.plan.pass[r.pi];
    const uint32_t lo = r.L - ps.b;
    const size_t c_lo = (size_t)1 << lo, c_out = r.cur_c < c_lo ? r.cur_c : c_lo, n = r.outer * c_out * r.j->gap;
    GRAPE_REQUIRE(n < ((size_t)1 << 32) - 256, "fold: more than 2^32 outputs in one pass");
    total = (uint32_t)n;
    out.out = fold_target(r, lo == 0);
    out.in = r.src;
    out.wts = r.wts + (size_t)fr26::N * ((size_t)r.pi << kFoldMaxBits);
    out.n_hi_max = (uint32_t)((r.cur_c + c_lo - 1) / c_lo);
    out.outer = (uint32_t)r.outer;
    out.c = (uint32_t)r.cur_c;
    out.lg_c_lo = lo;
    out.gap = r.j->gap;
    r.src = out.out;
    r.cur_c = c_out;
    r.L = lo;
    r.pi++;
    r.ints = false;                    // the first pass of a fold of integers leaves field elements
    return GRAPE_OK;
}

extern "C++" {
template <bool I32>
static void launch_fold_pass(const FoldPassArgs& a, uint32_t P, unsigned blocks, hipStream_t s) {
    if (P == 1) fold_pass_kernel<1, I32><<<blocks, kBlock, 0, s>>>(a);
    else if (P == 2) fold_pass_kernel<2, I32><<<blocks, kBlock, 0, s>>>(a);
    else if (P == 4) fold_pass_kernel<4, I32><<<blocks, kBlock, 0, s>>>(a);
    else if (P == 16) fold_short_kernel<16, I32><<<blocks, kBlock, 0, s>>>(a);
    else fold_short_kernel<256, I32><<<blocks, kBlock, 0, s>>>(a);
}
}

// Folds of up to two tensors, pass by pass; passes of one kind that stand at the same place of both share a launch.  Two operands of
// a matrix product go through the same kinds of passes: 32 heads of 2048 x 128 integers took two chains of four
// launches, 100 us of kernels, and take one of three, 41 (the proof 172 -> 113 us).
static int fold_jobs(const grape_fold_job* jobs, uint32_t count, grape_stream_t st) {
    hipStream_t s = as_stream(st);
    FoldRun run[kFoldJobs];
    FoldWeights fw = {};
    size_t scratch = 0;
    for (uint32_t k = 0; k < count; k++) {
        int rc = fold_start(run[k], jobs[k], count == 1, s);
        if (rc) return rc;
        if (run[k].done) continue;
        scratch += 2 * run[k].each;
        fw.x[k] = jobs[k].x;
        if (run[k].ints && run[k].plan.npass) fw.plain |= 1u << fw.npass;
        for (uint32_t i = 0; i < run[k].plan.npass; i++, fw.npass++) {
            fw.lo[fw.npass] = run[k].plan.lo[i];
            fw.b[fw.npass] = run[k].plan.pass[i].b;
        }
        if (k == 0) fw.npass0 = fw.npass;
    }
    if (scratch) {
        void* p;
        int rc = scratch_get(kSlotFold, scratch * 32 + 64, &p, s);
        if (rc) return rc;
        uint32_t* ws = (uint32_t*)p;
        for (uint32_t k = 0; k < count; k++) {
            for (int i = 0; i < 2; i++, ws += 8 * run[k].each) run[k].ws[i] = ws;
        }
    }
    if (fw.npass) {
        void* p;
        int rc = scratch_get(kSlotFoldW, ((size_t)kFoldJobs * kFoldMaxPasses * (1u << kFoldMaxBits) + 64) * fr26::N * 4, &p, s);
        if (rc) return rc;
        profile_begin();
        profile_mark(s);
        fold_weights_kernel<<<fw.npass, kBlock, 0, s>>>((int32_t*)p, fw);
        GRAPE_LAUNCH_CHECK();
        profile_mark(s);               // profiled intervals: the weight kernel, then one per pass
        run[0].wts = (const int32_t*)p;
        if (count > 1) run[1].wts = (const int32_t*)p + ((size_t)fr26::N * fw.npass0 << kFoldMaxBits);
    }
    auto at_pass = [&](uint32_t k) { return !run[k].done && run[k].pi < run[k].plan.npass; };
    for (;;) {
        FoldPassArgs a = {};
        unsigned blocks = 0;
        uint32_t P = 0, jobs_in = 0;
        bool plain = false;
        for (uint32_t k = 0; k < count; k++) {
            if (!at_pass(k)) continue;
            const uint32_t pk = run[k].plan.pass[run[k].pi].P;
            if (jobs_in && (pk != P || run[k].ints != plain)) continue;        // takes the next launch
            P = pk;
            plain = run[k].ints;
            uint32_t total = 0;
            int rc = fold_next(run[k], a.job[jobs_in++], total);
            if (rc) return rc;
            if (jobs_in == 1) a.blocks0 = 0xffffffffu;
            else a.blocks0 = blocks;
            blocks += blocks_for(total, kBlock / (int)P);
        }
        if (!jobs_in) break;
        if (plain) launch_fold_pass<true>(a, P, blocks, s);
        else launch_fold_pass<false>(a, P, blocks, s);
        GRAPE_LAUNCH_CHECK();
        profile_mark(s);
    }
    for (uint32_t k = 0; k < count; k++) {
        FoldRun& r = run[k];
        if (r.done) continue;
        if (r.plan.npass == 0) {
            // reading slabs o*c*gap of t while writing o*gap of it would race across workgroups: through scratch
            uint32_t* dst = fold_target(r, true);
            fold_small_kernel<<<(unsigned)r.outer, kBlock, 0, s>>>(dst, r.src, r.j->x + 8 * (size_t)r.j->id, r.L, r.cur_c, r.j->gap);
            GRAPE_LAUNCH_CHECK();
            r.src = dst;
        }
        if (r.src != r.j->t) GRAPE_HIP_CHECK(hipMemcpyAsync(r.j->t, r.src, r.outer * r.j->gap * 32, hipMemcpyDeviceToDevice, s));
    }
    return GRAPE_OK;
}

int grape_fr_random(uint32_t* out, size_t n, const uint32_t* key, grape_stream_t st) {
    if (n == 0) return GRAPE_OK;
    CHECK_PTR16(out);
    GRAPE_REQUIRE(key != nullptr && n <= ((size_t)1 << 32), "a key of eight words (host), at most 2^32 elements");
    RandomKey k;
    for (int i = 0; i < 8; i++) k.w[i] = key[i];
    random_kernel<<<blocks_for(n, 64), 64, 0, as_stream(st)>>>(out, n, k);
    GRAPE_LAUNCH_CHECK();
    return GRAPE_OK;
}

int grape_fr_fold(uint32_t* t, size_t N, const uint32_t* x, uint32_t c, uint32_t id, uint32_t gap, grape_stream_t st) {
    const grape_fold_job j = {t, nullptr, nullptr, N, x, c, id, gap};
    return fold_jobs(&j, 1, st);
}
int grape_fr_fold_from(uint32_t* out, const uint32_t* in, size_t N, const uint32_t* x, uint32_t c, uint32_t id, uint32_t gap, grape_stream_t st) {
    if (N == 0) return GRAPE_OK;
    CHECK_PTR16(in);
    const grape_fold_job j = {out, in, nullptr, N, x, c, id, gap};
    return fold_jobs(&j, 1, st);
}

size_t grape_fr_fold_i32_elems(size_t N, uint32_t c, uint32_t gap) {
    if (N == 0 || c == 0 || gap == 0 || N % ((size_t)c * gap) != 0) return N;
    const size_t outer = N / ((size_t)c * gap);
    size_t most = 0;
    for (const bool ints : {false, true}) {            // integers are folded in other steps than field elements
        FoldPlan plan;
        if (plan_fold(outer, c, gap, 0, ints, true, plan) != GRAPE_OK || plan.npass == 0) return N;
        const size_t c_lo = (size_t)1 << (log2ceil(c) - plan.pass[0].b);
        // several outer indices: the passes go through work memory of the library; one: the first pass writes into d_out
        const size_t n = outer > 1 ? outer * gap : (c < c_lo ? c : c_lo) * gap;
        if (n > most) most = n;
    }
    return most;
}

int grape_fr_fold_i32(uint32_t* out, const int32_t* in, size_t N, const uint32_t* x, uint32_t c, uint32_t id, uint32_t gap, grape_stream_t st) {
    GRAPE_REQUIRE(in != nullptr || N == 0, "null input");
    const grape_fold_job j = {out, nullptr, in, N, x, c, id, gap};
    return fold_jobs(&j, 1, st);
}

int grape_fr_fold_pair(const grape_fold_job* jobs, uint32_t count, grape_stream_t st) {
    GRAPE_REQUIRE(jobs != nullptr && count >= 1 && count <= (uint32_t)kFoldJobs, "one or two folds");
    return fold_jobs(jobs, count, st);
}

}  // extern "C"
