#include "prove.hpp"
#include "carried.hpp"
#include <algorithm>
#include <cassert>
#include <memory>
#include "../../include/grape_hip.h"

using grape_host::check;
using grape_host::OnDefaultStream;
static inline uint32_t* W(fr_t* p) { return reinterpret_cast<uint32_t*>(p); }
static inline const uint32_t* W(const fr_t* p) { return reinterpret_cast<const uint32_t*>(p); }

static void record(SumcheckTranscript* t, const Polynomial& p, const Fr& claim) {
    if (t) {
        t->rounds.push_back(p);
        t->claims.push_back(claim);
    }
}
static void read3(fr_t* d_sums, Fr out[3]) {
    check(grape_memcpy_d2h(out, d_sums, 3 * sizeof(fr_t), nullptr), "grape_memcpy_d2h");
}

namespace {
constexpr uint kLongRoundPairs = 1u << 16;       // from here on a round folds through the table of its challenge's multiples
constexpr uint kCarriedRow = 256;                // shortest row of an element product that carries its weights
constexpr uint kSplitLow = GRAPE_EQ_SPLIT_LOW, kLongestPrefix = GRAPE_EQ_LONGEST_PREFIX;
// device buffer released on scope exit
struct DeviceBuf {
    void* p = nullptr;
    explicit DeviceBuf(size_t bytes) { check(grape_malloc_on_default(&p, bytes ? bytes : 1), "grape_malloc"); }
    ~DeviceBuf() { grape_free_on_default(p); }
    DeviceBuf(const DeviceBuf&) = delete;
    DeviceBuf& operator=(const DeviceBuf&) = delete;
    fr_t* fr() const { return static_cast<fr_t*>(p); }
};
// eq tables of every prefix of `nvars` device challenges starting at d_u (level j at offset 2^j - 1)
struct EqPyramid {
    DeviceBuf buf;
    EqPyramid(const fr_t* d_u, uint nvars) : buf(sizeof(fr_t) * grape_eq_pyramid_elems(nvars)) {
        check(grape_eq_pyramid(W(buf.fr()), reinterpret_cast<const uint32_t*>(d_u), nvars, nullptr), "grape_eq_pyramid");
    }
    fr_t* level(uint j) const { return buf.fr() + (((size_t)1 << j) - 1); }
};
// Weights of the rounds of a long sumcheck over nvars variables at d_u: tables of every prefix as far as `whole` variables; longer
// rounds take their weight as a product of a table over the lowest `low` variables and one over the rest.
struct EqWeights {
    uint low, whole;
    EqPyramid prefix;
    std::unique_ptr<EqPyramid> high;
    EqWeights(const fr_t* d_u, uint nvars, uint low_, uint whole_) : low(low_), whole(std::min(nvars, whole_)), prefix(d_u, whole) {
        if (nvars > whole) high.reset(new EqPyramid(d_u + low, nvars - low));
    }
    void weigh(grape_wround_args& a, uint vars, uint period) const {
        a.eq = W(prefix.level(vars > whole ? low : vars));
        a.eq_high = vars > whole ? W(high->level(vars - low)) : nullptr;
        a.period = period;
    }
};
std::vector<Fr> download_vec(const fr_t* d, size_t n) {
    std::vector<Fr> out(n);
    if (n) check(grape_memcpy_d2h(out.data(), d, sizeof(fr_t) * n, nullptr), "grape_memcpy_d2h");
    return out;
}
}  // namespace

// Phase 1 of the matmul sumcheck (src/prove.cu:49-85) binds the batch variables l of
// sum_l eq(u_l, l) sum_k A[l][k] B[l][k].  The reference writes three coefficient arrays per round,
// folds each over the remaining l-bits of u and sums the K survivors; here every round is one
// launch that folds A and B and takes the three sums per batch row, weighted by that row's
// eq(u_low, l') from a table built once.  The rounds are queued back to back (the challenges
// are known up front) and their sums read with one copy.
Fr matmul_sumcheck_phase1(FrTensor& A, FrTensor& B, FrTensor& a, FrTensor& b, FrTensor& c, fr_t* u, fr_t* v, uint K, uint size,
                          Fr& claim, SumcheckTranscript* transcript) {
    (void)a;
    (void)b;
    (void)c;
    const uint rounds = Log2(size / K);
    Fr eq_accumulate = Fr::one();
    if (rounds == 0) return eq_accumulate;
    if (size != (K << rounds)) throw std::runtime_error("matmul_phase1: the batch extent must be a power of two");
    const std::vector<Fr> us = download_vec(u - rounds, rounds), vs = download_vec(v - rounds, rounds);
    EqPyramid eq(u - rounds, rounds - 1);
    FrTensor sums(3 * rounds, OnDefaultStream());
    uint in = size;
    for (uint i = 0; i < rounds; i++) {
        const uint out = in / 2;
        check(grape_sumcheck_round2_seg(W(A.gpu_data), W(B.gpu_data), in, out, K, W(eq.level(rounds - 1 - i)), W(v - i - 1),
                                        W(sums.gpu_data + 3 * i), nullptr),
              "grape_sumcheck_round2_seg");
        in = out;
    }
    const std::vector<Fr> s = download_vec(sums.gpu_data, 3 * (size_t)rounds);
    for (uint i = 0; i < rounds; i++) {
        const Fr &u_now = us[rounds - 1 - i], &v_now = vs[rounds - 1 - i];
        Polynomial p({s[3 * i], s[3 * i + 1], s[3 * i + 2]});
        p *= (Polynomial::eq(u_now) * eq_accumulate);
        if (p(0) + p(1) != claim) throw std::runtime_error("matmul_phase1: claim != p(0) + p(1)");
        claim = p(v_now);
        record(transcript, p, claim);
        eq_accumulate *= Polynomial::eq(u_now, v_now);
    }
    return eq_accumulate;
}

// rounds of at least this many index pairs take their middle coefficient from the running claim
static constexpr uint kClaimRoundMinOut = 1u << 16;

// src/prove.cu:87-117, with the three reductions fused into the round kernel
void matmul_sumcheck_phase2(FrTensor& A, FrTensor& B, FrTensor& a, FrTensor& b, FrTensor& c, fr_t* v, uint K, Fr& claim,
                            Fr& eq_accumulate, SumcheckTranscript* transcript) {
    (void)a;
    (void)b;
    (void)c;
    uint rounds = Log2(K);
    if (rounds == 0) return;
    uint inputsize = K;
    uint outputsize = 1u << (rounds - 1);
    // all challenges of this phase in one copy
    std::vector<Fr> vs(rounds);
    check(grape_memcpy_d2h(vs.data(), v - rounds, sizeof(fr_t) * rounds, nullptr), "grape_memcpy_d2h");
    // The challenges are known before the first round, so all rounds are queued back to back,
    // each leaving its three sums in its own slot, and read with one copy at the end (the
    // reference copies and synchronises after every round).
    FrTensor sums(3 * rounds, OnDefaultStream());
    // Long rounds (2^16 index pairs and more) are bound by their limb products, and one of the three
    // per pair can go when the round is given the running claim: p(0) + p(1) = claim fixes the middle
    // coefficient.  The claim the kernels chain is the one of the bare sums (without eq_accumulate).
    fr_t* d_claim = nullptr;
    if (outputsize >= kClaimRoundMinOut && !(eq_accumulate == Fr::zero())) {
        d_claim = grape_host::upload(std::vector<Fr>{claim * eq_accumulate.inverse()}, OnDefaultStream());
    }
    struct Release {
        fr_t*& p;
        ~Release() { grape_free_on_default(p); }
    } release{d_claim};
    for (uint i = 0; i < rounds; i++) {
        if (d_claim && outputsize >= kClaimRoundMinOut) {
            check(grape_sumcheck_round2_claim(W(A.gpu_data), W(B.gpu_data), inputsize, outputsize, W(v - i - 1), W(d_claim),
                                              W(sums.gpu_data + 3 * i), nullptr),
                  "grape_sumcheck_round2_claim");
            inputsize = outputsize;
            outputsize = outputsize / 2;
            continue;
        }
        if (inputsize <= 512) {
            // short tensors: all remaining rounds in one launch
            check(grape_sumcheck_round2_tail(W(A.gpu_data), W(B.gpu_data), inputsize, rounds - i, W(v - i), W(sums.gpu_data + 3 * i), nullptr),
                  "grape_sumcheck_round2_tail");
            break;
        }
        check(grape_sumcheck_round2(W(A.gpu_data), W(B.gpu_data), inputsize, outputsize, W(v - i - 1), W(sums.gpu_data + 3 * i), nullptr),
              "grape_sumcheck_round2");
        inputsize = outputsize;
        outputsize = outputsize / 2;
    }
    std::vector<Fr> s(3 * (size_t)rounds);
    check(grape_memcpy_d2h(s.data(), sums.gpu_data, sizeof(fr_t) * 3 * rounds, nullptr), "grape_memcpy_d2h");
    for (uint i = 0; i < rounds; i++) {
        Polynomial p({s[3 * i] * eq_accumulate, s[3 * i + 1] * eq_accumulate, s[3 * i + 2] * eq_accumulate});
        if (p(0) + p(1) != claim) throw std::runtime_error("matmul_phase2: claim != p(0) + p(1)");
        const Fr& v_now = vs[rounds - 1 - i];
        claim = p(v_now);
        record(transcript, p, claim);
    }
}

namespace {
// An operand of prove_matmul: a tensor that the proof consumes, or a tensor of field elements or of integers (read as
// FrTensor::get_data would embed them) that is kept - the fold over its row variables, which reads it once, reads it in place.
struct Operand {
    FrTensor* consumed = nullptr;
    const fr_t* kept = nullptr;
    const int* ints = nullptr;
    std::unique_ptr<FrTensor> own;
    // the fold over the row variables, into a tensor of its own where the operand is kept
    grape_fold_job fold(uint size, fr_t* x, uint c, uint id, uint gap) {
        if (!consumed) {
            own.reset(new FrTensor((uint)std::max<size_t>(grape_fr_fold_i32_elems(size, c, gap), 1), OnDefaultStream()));
            own->set_size(size / (c * gap) * gap);
        }
        grape_fold_job j{};
        j.t = W(tensor().gpu_data);
        if (kept) j.from = W(kept);
        j.ints = ints;
        j.N = size;
        j.x = W(x);
        j.c = c;
        j.id = id;
        j.gap = gap;
        return j;
    }
    FrTensor& tensor() { return consumed ? *consumed : *own; }
};
// Both phases where the folded operands are short: all rounds in one call, and one copy brings their sums and the two
// elements that are left.  u, v (host) and U, V (device) point behind the variables of the batch and inner index.
std::pair<Fr, Fr> matmul_short_rounds(FrTensor& A, FrTensor& B, int L, int K, const Fr* u, const Fr* v, const fr_t* U, const fr_t* V, Fr& claim,
                                      Fr& eq_accumulate, SumcheckTranscript* transcript) {
    const uint phase1 = Log2((uint)L), rounds = phase1 + Log2((uint)K);
    FrTensor sums(3 * rounds + 2, OnDefaultStream());
    grape_short_rounds_args a{};
    a.kind = GRAPE_SHORT_PAIR;
    a.size = (uint)L * (uint)K;
    a.row = (uint)K;
    a.v_end = W(V);
    a.sums = W(sums.gpu_data);
    a.stride = 3;
    FrTensor* const x[2] = {&A, &B};
    for (uint k = 0; k < 2; k++) {
        a.x[k] = a.last[k] = W(x[k]->gpu_data);
        a.last_copy[k] = W(sums.gpu_data + 3 * rounds + k);
    }
    std::unique_ptr<EqPyramid> eq;
    if (phase1) {
        eq.reset(new EqPyramid(U - phase1, phase1 - 1));
        a.weights = GRAPE_SHORT_ROWS;
        a.pyramid = W(eq->level(0));
        a.top_level = phase1 - 1;
    }
    check(grape_short_rounds(&a, nullptr), "grape_short_rounds");
    const std::vector<Fr> s = download_vec(sums.gpu_data, 3 * (size_t)rounds + 2);
    eq_accumulate = Fr::one();
    for (uint i = 0; i < rounds; i++) {
        const Fr& v_now = *(v - 1 - i);
        Polynomial p;
        if (i < phase1) {
            const Fr& u_now = *(u - 1 - i);
            p = Polynomial({s[3 * i], s[3 * i + 1], s[3 * i + 2]});
            p *= (Polynomial::eq(u_now) * eq_accumulate);
            if (p(0) + p(1) != claim) throw std::runtime_error("matmul_phase1: claim != p(0) + p(1)");
            eq_accumulate *= Polynomial::eq(u_now, v_now);
        } else {
            p = Polynomial({s[3 * i] * eq_accumulate, s[3 * i + 1] * eq_accumulate, s[3 * i + 2] * eq_accumulate});
            if (p(0) + p(1) != claim) throw std::runtime_error("matmul_phase2: claim != p(0) + p(1)");
        }
        claim = p(v_now);
        record(transcript, p, claim);
    }
    return {s[3 * (size_t)rounds], s[3 * (size_t)rounds + 1]};
}
std::pair<Fr, Fr> prove_matmul_impl(Operand A_op, Operand B_op, int L, int N, int M, int K, const std::vector<Fr>& u, const std::vector<Fr>& v,
                                    Fr& claim, SumcheckTranscript* transcript) {
    // The point u is read as log2(M) variables of the column index, log2(N) of the row index and log2(L)
    // of the batch index, while the reference finds the end of the batch variables at Log2(L*N*M)
    // (src/prove.cu:198): the two agree only when the padded extents multiply to the padded product.
    // A shape like N = 3, M = 5 (Log2(15) = 4, but 2 + 3 variables) has no defined reading - the
    // reference's folds would run past the end of u - and is refused, as is a point that is too short.
    const uint lu = Log2((uint)L) + Log2((uint)N) + Log2((uint)M);
    if (L < 1 || N < 1 || M < 1 || K < 1 || Log2((uint)(L * N * M)) != lu || u.size() < lu || v.size() < Log2((uint)(L * K)))
        throw std::runtime_error("prove_matmul: Incompatible dimensions");
    fr_t* U = grape_host::upload(u, OnDefaultStream());
    fr_t* V = grape_host::upload(v, OnDefaultStream());
    std::pair<Fr, Fr> ret;
    try {
        const grape_fold_job folds[2] = {A_op.fold((uint)(L * N * K), U, N, Log2(M), K), B_op.fold((uint)(L * M * K), U, M, 0, K)};
        // one tensor as both operands is folded twice, one fold after the other
        const bool apart = folds[0].t != folds[1].t;
        check(grape_fr_fold_pair(folds, apart ? 2 : 1, nullptr), "grape_fr_fold_pair");
        if (!apart) check(grape_fr_fold_pair(folds + 1, 1, nullptr), "grape_fr_fold_pair");
        FrTensor &A = A_op.tensor(), &B = B_op.tensor();
        Fr eq_accumulate;
        if ((uint)(L * K) >= 2 && (uint)(L * K) <= GRAPE_SHORT_MAX && (L & (L - 1)) == 0) {
            ret = matmul_short_rounds(A, B, L, K, u.data() + Log2(L * N * M), v.data() + Log2(L * K), U + Log2(L * N * M), V + Log2(L * K), claim,
                                      eq_accumulate, transcript);
        } else {
            FrTensor a(1, OnDefaultStream()), b(1, OnDefaultStream()), c(1, OnDefaultStream());      // the reference's coefficient arrays (src/prove.cu:190-192): not used by the fused rounds
            eq_accumulate = matmul_sumcheck_phase1(A, B, a, b, c, U + Log2(L * N * M), V + Log2(L * K), K, K * L, claim, transcript);
            matmul_sumcheck_phase2(A, B, a, b, c, V + Log2(K), K, claim, eq_accumulate, transcript);
            ret.first = grape_host::download(A.gpu_data);
            ret.second = grape_host::download(B.gpu_data);
        }
        if (ret.first * ret.second * eq_accumulate != claim) throw std::runtime_error("prove_matmul: A(v) * B(v) * eq != claim");
    } catch (...) {
        grape_free_on_default(V);
        grape_free_on_default(U);
        throw;
    }
    grape_free_on_default(V);
    grape_free_on_default(U);
    return ret;
}
}  // namespace

// src/prove.cu:175-210
std::pair<Fr, Fr> prove_matmul(FrTensor& A, FrTensor& B, int L, int N, int M, int K, const std::vector<Fr> u,
                               const std::vector<Fr> v, Fr& claim, SumcheckTranscript* transcript) {
    Operand a, b;
    a.consumed = &A;
    b.consumed = &B;
    return prove_matmul_impl(std::move(a), std::move(b), L, N, M, K, u, v, claim, transcript);
}
std::pair<Fr, Fr> prove_matmul(const fr_t* device_A, const fr_t* device_B, int L, int N, int M, int K, const std::vector<Fr> u,
                               const std::vector<Fr> v, Fr& claim, SumcheckTranscript* transcript) {
    Operand a, b;
    a.kept = device_A;
    b.kept = device_B;
    return prove_matmul_impl(std::move(a), std::move(b), L, N, M, K, u, v, claim, transcript);
}
std::pair<Fr, Fr> prove_matmul(const int* device_int_A, const int* device_int_B, int L, int N, int M, int K, const std::vector<Fr> u,
                               const std::vector<Fr> v, Fr& claim, SumcheckTranscript* transcript) {
    Operand a, b;
    a.ints = device_int_A;
    b.ints = device_int_B;
    return prove_matmul_impl(std::move(a), std::move(b), L, N, M, K, u, v, claim, transcript);
}

// The element-product sumcheck (src/prove.cu:119-172) proves sum_x eq(u, x) A(x) B(x) over tensors
// of first_size rows of second_size = size / first_size elements, the row index bound first
// (rows are not padded; a last row extent that is no power of two reads as zero-extended).  The
// reference writes three coefficient arrays per round and folds each over the remaining variables
// of u; here a round is one launch that folds A and B and takes the three sums weighted by
// eq(u_low, x) from a pyramid of tables built once - on rows padded to a power of two, which is
// where the variables of u live.
// A and B are read by the first round, every round leaves its folded halves in Aw and Bw (A and B themselves, or
// buffers of size / 2 elements where the operands are kept).  u and v (device) point behind the variables, as do hu and hv (host; where
// the caller has no host copy they are downloaded).  The elements that are left go to claims where that is given.
static Fr eleMul_rounds(fr_t* Aw, fr_t* Bw, const fr_t* A, const fr_t* B, fr_t* u, fr_t* v, const Fr* hu, const Fr* hv, uint first_size, uint size,
                        Fr& claim, std::pair<Fr, Fr>* claims, SumcheckTranscript* transcript) {
    if ((1u << Log2(first_size)) != first_size) throw std::runtime_error("eleMul_sumcheck: first_size is illegal");
    const uint second_size = size / first_size;
    const uint rounds = Log2(size);
    Fr eq_accumulate = Fr::one();
    if (rounds == 0) {
        if (claims) *claims = {grape_host::download(A), grape_host::download(B)};
        return eq_accumulate;
    }
    const uint row_pad = 1u << Log2(second_size);
    std::vector<Fr> us, vs;
    if (!hu) {
        us = download_vec(u - rounds, rounds);
        vs = download_vec(v - rounds, rounds);
        hu = us.data() + rounds;
        hv = vs.data() + rounds;
    }
    // Long rounds: the weights of a padded row split into row and column, those of whole powers of two at 2^kSplitLow.  A row whose
    // padded length has no prefix table of its own (above 2^20) is weighed by whole tables.
    const uint lg_row = Log2(second_size);
    const bool padded = second_size != row_pad;
    const uint low = padded ? lg_row : kSplitLow;
    FrTensor sums(3 * rounds + 2, OnDefaultStream());
    // the tables of all challenges' multiples, and every long round's partial sums until one launch finishes them all
    std::vector<grape_wround_args> queued;
    std::vector<std::unique_ptr<DeviceBuf>> partials;
    std::unique_ptr<DeviceBuf> tabs;
    if (size / 2 >= kLongRoundPairs) {
        tabs.reset(new DeviceBuf(sizeof(int32_t) * GRAPE_FOLD_TABLE_WORDS * (size_t)rounds));
        check(grape_fold_tables(static_cast<int32_t*>(tabs->p), W(v - rounds), rounds, nullptr), "grape_fold_tables");
    }
    uint in = size, out = size / 2;
    // The leading long rounds that pair whole rows (whole powers of two) carry their weights in B from the first one on, from 2^20
    // pairs: 0.39 ms either way there, while 2^18 elements take 0.225 against 0.210 ms (an upload, two launches for tables, one
    // to end) and 1024 x 11008 take 0.82 against 0.96.
    // What is left in B takes a factor per row, made here and uploaded: rows of kCarriedRow elements leave fewer than 512 (2^13 x 257:
    // 0.41-0.43 against 0.45 ms, 2^16 x 257: 1.10 against 1.30), rows of 5 would leave 2^14.
    // A tensor times itself, bound in place, has one buffer for both folds: its long rounds fail their check, and carried ones would not.
    const uint period = padded ? second_size : 1u << kSplitLow;
    uint carrying = 0;
    if (Aw != Bw && period >= kCarriedRow && period <= GRAPE_WROUND_MAX_PERIOD && size / 2 >= 1u << 20)
        for (uint n = size; n % 2 == 0 && n / 2 >= kLongRoundPairs && (n / 2) % period == 0; n /= 2) carrying++;
    const CarriedFactors factors(hu - rounds, hv - rounds, rounds, carrying, low);
    const bool carry = factors.ok && carrying >= 2;
    // carried rounds read the split tables alone, and the rounds behind them a prefix table of at most 2^kSplitLow entries or a split one;
    // four rows and more leave variables above both
    const EqWeights eq(u - rounds, rounds - 1, low, carry ? std::max(low, kSplitLow) : padded && lg_row > kLongestPrefix ? rounds : kLongestPrefix);
    std::vector<grape_carried_args> carried;
    std::unique_ptr<DeviceBuf> consts, ratio_tabs;
    if (carry) {
        std::vector<Fr> c(factors.ratio);
        c.insert(c.end(), factors.end.begin(), factors.end.end());
        consts.reset(new DeviceBuf(sizeof(fr_t) * c.size()));
        check(grape_memcpy_h2d(consts->p, c.data(), sizeof(fr_t) * c.size(), nullptr), "grape_memcpy_h2d");
        ratio_tabs.reset(new DeviceBuf(sizeof(int32_t) * GRAPE_FOLD_TABLE_WORDS * (size_t)carrying));
        check(grape_fold_tables(static_cast<int32_t*>(ratio_tabs->p), W(consts->fr()), carrying, nullptr), "grape_fold_tables");
        for (uint i = 0; i < carrying; i++, in = out, out /= 2) {
            grape_carried_args a{};
            a.A_out = W(Aw);
            a.Z_out = W(Bw);
            a.A = W(i ? Aw : A);
            a.Z = W(i ? Bw : B);
            a.eq = W(eq.prefix.level(low));
            a.eq_high = i == 0 ? W(eq.high->level(rounds - 1 - low)) : nullptr;
            a.period = period;
            a.n_out = out;
            a.tab_a = static_cast<int32_t*>(tabs->p) + (size_t)GRAPE_FOLD_TABLE_WORDS * (rounds - 1 - i);
            a.tab_z = static_cast<int32_t*>(ratio_tabs->p) + (size_t)GRAPE_FOLD_TABLE_WORDS * i;
            carried.push_back(a);
        }
        for (uint i = 0; i < carrying; i++) {
            carried[i].pair = CarriedFactors::place_in_pass(i, carrying);
            partials.emplace_back(new DeviceBuf(grape_carried_partial_bytes(&carried[i])));
            carried[i].partial = W(partials.back()->fr());
        }
        CarriedFactors::queue_passes(carried.data(), carrying, nullptr);
        check(grape_carried_finish(W(sums.gpu_data), 3, carried.data(), carrying, nullptr), "grape_carried_finish");
        check(grape_carried_end(W(Bw), W(Bw), in, W(consts->fr() + carrying), period, nullptr, nullptr), "grape_carried_end");
        if (in == second_size) out = 1u << (Log2(in) - 1);     // a row's own variables: those of its padded length
    }
    const uint done = (uint)carried.size();
    for (uint i = done; i < rounds; i++) {
        const fr_t *Ai = i ? Aw : A, *Bi = i ? Bw : B;
        // short rounds in one call; a single row that is no power of two has no defined first round and is refused below
        if (in <= GRAPE_SHORT_MAX && out < kLongRoundPairs && ((in & (in - 1)) == 0 || (first_size > 1 && in % second_size == 0))) {
            grape_short_rounds_args a{};
            a.kind = GRAPE_SHORT_PAIR;
            a.weights = GRAPE_SHORT_FULL;
            a.size = in;
            a.row = in < second_size ? in : second_size;
            a.x[0] = W(Ai);
            a.x[1] = W(Bi);
            a.v_end = W(v - i);
            a.pyramid = W(eq.prefix.level(0));
            a.top_level = rounds - 1 - i;
            a.sums = W(sums.gpu_data + 3 * i);
            a.stride = 3;
            a.last[0] = W(Aw);
            a.last[1] = W(Bw);
            a.last_copy[0] = W(sums.gpu_data + 3 * rounds);
            a.last_copy[1] = W(sums.gpu_data + 3 * rounds + 1);
            check(grape_short_rounds(&a, nullptr), "grape_short_rounds");
            break;
        }
        // while whole rows are paired the weights are addressed on padded rows
        const bool rows = in > second_size && padded;
        grape_wround_args a{};
        a.A_out = W(Aw);
        a.S_out = W(Bw);
        a.A = W(Ai);
        a.S = W(Bi);
        eq.weigh(a, rounds - 1 - i, rows ? second_size : 1u << kSplitLow);
        a.rowlen = rows ? second_size : 1;
        a.rowpad = rows ? row_pad : 1;
        a.in_size = in;
        a.n_out = out;
        a.v = W(v - i - 1);
        a.tab = out >= kLongRoundPairs ? static_cast<int32_t*>(tabs->p) + (size_t)GRAPE_FOLD_TABLE_WORDS * (rounds - 1 - i) : nullptr;
        partials.emplace_back(new DeviceBuf(grape_wround_partial_bytes(&a)));
        a.partial = W(partials.back()->fr());
        check(grape_wround_queue(&a, nullptr), "grape_wround_queue");
        queued.push_back(a);
        in = out;
        out = out == second_size ? (1u << (Log2(out) - 1)) : out / 2;
        if (out == 0) out = 1;
    }
    if (!queued.empty()) check(grape_wround_finish(W(sums.gpu_data + 3 * (size_t)done), 3, queued.data(), (uint)queued.size(), nullptr), "grape_wround_finish");
    std::vector<Fr> s = download_vec(sums.gpu_data, 3 * (size_t)rounds + 2);
    for (uint i = done; i-- > 0;) {
        Fr* c = &s[3 * (size_t)i];
        const std::array<Fr, 3> q = factors.polynomial(i, c[0] * factors.at0[i], c[1] * factors.at1[i], c[3], c[3] + c[4] + c[5]);
        std::copy(q.begin(), q.end(), c);
    }
    for (uint i = 0; i < rounds; i++) {
        const Fr &u_now = *(hu - 1 - i), &v_now = *(hv - 1 - i);
        Polynomial p({s[3 * i], s[3 * i + 1], s[3 * i + 2]});
        p *= (Polynomial::eq(u_now) * eq_accumulate);
        if (p(0) + p(1) != claim) throw std::runtime_error("ele_Mul: claim != p(0) + p(1)");
        claim = p(v_now);
        record(transcript, p, claim);
        eq_accumulate *= Polynomial::eq(u_now, v_now);
    }
    if (claims) *claims = {s[3 * (size_t)rounds], s[3 * (size_t)rounds + 1]};
    return eq_accumulate;
}

Fr eleMul_sumcheck(FrTensor& A, FrTensor& B, FrTensor& a, FrTensor& b, FrTensor& c, fr_t* u, fr_t* v, uint first_size, uint size,
                   Fr& claim, SumcheckTranscript* transcript) {
    (void)a;
    (void)b;
    (void)c;
    return eleMul_rounds(A.gpu_data, B.gpu_data, A.gpu_data, B.gpu_data, u, v, nullptr, nullptr, first_size, size, claim, nullptr, transcript);
}

static std::pair<Fr, Fr> prove_eleMul_impl(fr_t* Aw, fr_t* Bw, const fr_t* A, const fr_t* B, int L, int M, int N, const std::vector<Fr>& u,
                                           const std::vector<Fr>& v, Fr& claim, SumcheckTranscript* transcript) {
    fr_t* U = grape_host::upload(u, OnDefaultStream());
    fr_t* V = grape_host::upload(v, OnDefaultStream());
    std::pair<Fr, Fr> ret;
    try {
        const uint size = (uint)(L * M * N);
        const uint lg = Log2(size);
        if (u.size() < lg || v.size() < lg) throw std::runtime_error("prove_eleMul: the point has too few variables");
        Fr eq_accumulate = eleMul_rounds(Aw, Bw, A, B, U + lg, V + lg, u.data() + lg, v.data() + lg, (uint)(L * M), size, claim, &ret, transcript);
        if (ret.first * ret.second * eq_accumulate != claim) throw std::runtime_error("prove_eleMul: A(v) * B(v) * eq != claim");
    } catch (...) {
        grape_free_on_default(V);
        grape_free_on_default(U);
        throw;
    }
    grape_free_on_default(V);
    grape_free_on_default(U);
    return ret;
}
// src/prove.cu:212-243
std::pair<Fr, Fr> prove_eleMul(FrTensor& A, FrTensor& B, int L, int M, int N, const std::vector<Fr> u, const std::vector<Fr> v,
                               Fr& claim, SumcheckTranscript* transcript) {
    return prove_eleMul_impl(A.gpu_data, B.gpu_data, A.gpu_data, B.gpu_data, L, M, N, u, v, claim, transcript);
}
std::pair<Fr, Fr> prove_eleMul(const fr_t* device_A, const fr_t* device_B, int L, int M, int N, const std::vector<Fr> u,
                               const std::vector<Fr> v, Fr& claim, SumcheckTranscript* transcript) {
    const uint size = (uint)(L * M * N);
    FrTensor Aw(size / 2 + 1, OnDefaultStream()), Bw(size / 2 + 1, OnDefaultStream());
    return prove_eleMul_impl(Aw.gpu_data, Bw.gpu_data, device_A, device_B, L, M, N, u, v, claim, transcript);
}

// combine_claims (src/prove.cu:245-300) merges several claims X(u_j) = claim_j about one tensor into
// one claim X(v) by a sumcheck over sum_j sum_x eq(u_j, x) X(x).  Per round the reference copies
// the two coefficient arrays once per claim and evaluates each copy at the remaining variables of
// u_j; here the weights of every claim come from its own eq pyramid (built once), one launch takes
// all 2*num weighted sums of the round from a single read of X per claim, a second folds X, and
// the rounds are queued without copies in between.
Fr combine_claims(FrTensor& X, const std::vector<Fr>& claims, const std::vector<std::vector<Fr>>& u, const std::vector<Fr>& v,
                  const uint size, SumcheckTranscript* transcript) {
    if (size != (1u << Log2(size))) throw std::runtime_error("combine_claims: size must be a power of two");
    const uint num = (uint)claims.size();
    for (uint i = 0; i < num; i++)
        if (u[i].size() != v.size()) throw std::runtime_error("combine_claims: point sizes differ");
    if ((1u << v.size()) != size) throw std::runtime_error("combine_claims: 2^|v| != size");
    Fr claim = Fr::zero();
    for (uint i = 0; i < num; i++) claim += claims[i];
    const uint rounds = (uint)v.size();
    std::vector<Fr> eq_accumulate(num, Fr::one());
    if (rounds > 0 && num > 0) {
        fr_t* d_v = grape_host::upload(v, OnDefaultStream());
        std::vector<std::unique_ptr<EqPyramid>> eq;
        std::vector<fr_t*> d_u(num, nullptr);
        FrTensor sums(2 * num * rounds, OnDefaultStream());
        try {
            for (uint j = 0; j < num; j++) {
                d_u[j] = grape_host::upload(u[j], OnDefaultStream());
                eq.emplace_back(new EqPyramid(d_u[j], rounds - 1));
            }
            uint in = size;
            for (uint i = 0; i < rounds; i++) {
                const uint out = in / 2;
                // one launch weighs the tensor against up to 16 tables: more claims go in groups of 16
                for (uint j0 = 0; j0 < num; j0 += 16) {
                    const uint nj = num - j0 < 16 ? num - j0 : 16;
                    const uint32_t* tables[16];
                    for (uint j = 0; j < nj; j++) tables[j] = W(eq[j0 + j]->level(rounds - 1 - i));
                    check(grape_wsum1_multi(W(X.gpu_data), tables, nj, in, out, W(sums.gpu_data + 2 * ((size_t)num * i + j0)), nullptr),
                          "grape_wsum1_multi");
                }
                uint32_t* ptrs[1] = {W(X.gpu_data)};
                check(grape_fr_fold_msb_multi(ptrs, 1, out, W(d_v + (rounds - 1 - i)), nullptr), "grape_fr_fold_msb_multi");
                in = out;
            }
            const std::vector<Fr> s = download_vec(sums.gpu_data, 2 * (size_t)num * rounds);
            for (uint i = 0; i < rounds; i++) {
                const Fr& v_now = v[rounds - 1 - i];
                Polynomial p(2);
                for (uint j = 0; j < num; j++) {
                    const Fr& now_u = u[j][rounds - 1 - i];
                    const Fr* sj = &s[2 * ((size_t)num * i + j)];
                    Polynomial p1({sj[0], sj[1]});
                    p1 *= Polynomial::eq(now_u);
                    p1 *= eq_accumulate[j];
                    p += p1;
                    eq_accumulate[j] *= Polynomial::eq(now_u, v_now);
                }
                if (p(0) + p(1) != claim) throw std::runtime_error("combine_claims: claim != p(0) + p(1)");
                claim = p(v_now);
                record(transcript, p, claim);
            }
        } catch (...) {
            check(grape_stream_sync(nullptr), "sync");
            for (fr_t* d : d_u) grape_free_on_default(d);
            grape_free_on_default(d_v);
            throw;
        }
        check(grape_stream_sync(nullptr), "sync");
        for (fr_t* d : d_u) grape_free_on_default(d);
        grape_free_on_default(d_v);
    }
    Fr ret = X(0u);
    Fr sum = Fr::zero();
    for (uint i = 0; i < num; i++) sum += eq_accumulate[i] * ret;
    if (sum != claim) throw std::runtime_error("combine_claims: final check failed");
    return ret;
}
