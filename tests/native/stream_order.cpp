// Programs against the host classes on the runtime of fake_hip.cpp: what is queued, waited for and refused.
// One scenario per run, named by the argument; exit status 0 when it holds.
#include <cstdio>
#include <cstring>
#include <functional>
#include <map>
#include <memory>
#include <string>
#include "../../include/grape_hip.h"
#include "../../grape_amd/host/host_capi.h"
#include "../../grape_amd/host/hyrax.hpp"
#include "../../grape_amd/host/prove.hpp"
#include "../../grape_amd/host/tlookup.hpp"

extern "C" {
unsigned long fake_pending(const void* stream);
unsigned long fake_unjoined();
unsigned long fake_launches();
unsigned long fake_launched(const char* part);
unsigned long fake_copies();
void fake_queue(const void* stream);
unsigned long fake_waits();
unsigned long fake_bytes();
void fake_limit(unsigned long bytes);
void fake_fail_launches(unsigned long n);
void fake_set_device(int device);
}

static int failures = 0;
static void expect(bool ok, const char* what) {
    if (!ok) {
        std::printf("does not hold: %s\n", what);
        failures++;
    }
}
static affine_t* device_points(size_t n) {
    void* p = nullptr;
    grape_host::ensure_init();
    grape_host::check(grape_malloc(&p, sizeof(affine_t) * n), "grape_malloc");
    return static_cast<affine_t*>(p);
}

// A range lookup whose proof is refused between its long rounds and its commitments (com_m has fewer rows than layers): the
// long rounds' sums are being finished on a stream of their own then, and everything they use is given back.
static void refused_lookup() {
    const uint D = 1u << 18, cols = 64, len = 256, layers = 64;
    bn128 G = bn128::one();
    Hyrax hyrax(layers, cols, device_points(256 * cols), G, 1);
    tLookupRange lookup(-128, len);
    FrTensor S(D), A(D);
    int* ints = reinterpret_cast<int*>(device_points(D / 16));
    double seconds = 0;
    std::string error;
    try {
        lookup.prove(ints, S, A, random_vec(18), hyrax, cols, seconds);
    } catch (const std::exception& e) {
        error = e.what();
    }
    expect(error.find("Size too small") == 0, "the commitment of the multiplicities is refused");
    expect(fake_unjoined() == 0, "no stream is left with work that nothing waits for");
}

// A proof that is refused for its arguments leaves nothing behind: the next one on the object, of field tensors in rows of 11008, has
// its witness compared with the table as on an object that has refused none.
static void proof_after_a_refused_one() {
    const uint rows = 16, D = rows * 11008, Dp = rows * 16384, cols = 64, len = 1024;
    bn128 G = bn128::one();
    Hyrax hyrax(1, cols, device_points(256 * cols), G, 1);
    const std::vector<int> map(len, 7);
    int* ints = reinterpret_cast<int*>(device_points(Dp / 8));
    double seconds = 0;
    auto proved = [&](const std::function<void()>& prove) {
        try {
            prove();
        } catch (const std::exception& e) {
            return std::string(e.what());
        }
        return std::string();
    };
    FrTensor A(Dp), S(Dp), S_out(D);
    S_out.set_size(D);
    tLookupRangeMapping mapping(-512, len, map.data());
    tLookupRange range(-512, len);
    auto compared = [&](bool is_mapping) {
        const unsigned long before = fake_launched("inverse_by_table");
        A.set_size(Dp);
        S.set_size(D);
        proved([&] {
            if (is_mapping) mapping.prove(S, S_out, A, random_vec(18), hyrax, cols, seconds);
            else range.prove(S, A, random_vec(18), hyrax, cols, seconds);
        });
        return fake_launched("inverse_by_table") - before;
    };
    expect(compared(true) == 1 && compared(false) == 1, "a padded witness of field elements is compared with the table");
    A.set_size(Dp);
    expect(proved([&] { mapping.prove(ints, ints, Dp, A, random_vec(17), hyrax, cols, seconds); }) == "u.size() != v.size()", "a mapping of integers is refused");
    S.set_size(Dp);
    expect(proved([&] { range.prove(ints, S, A, random_vec(17), hyrax, cols, seconds); }) == "u.size() != v.size()", "a range of integers is refused");
    expect(compared(true) == 1, "so it is after a mapping that was refused");
    expect(compared(false) == 1, "so it is after a range that was refused");
}

// Carried rounds gather two multiples of every table entry: made for tables of up to 2^24 entries, and no room is asked for beyond.
static void carried_lookups() {
    const uint cols = 64, gens = 1u << 15;                // the multiplicities are committed in rows of 2^(log_len / 2)
    bn128 G = bn128::one();
    Hyrax hyrax(1, gens, device_points(256 * (size_t)gens), G, 1);
    double seconds = 0;
    auto carried = [&](uint log_len, uint log_D) {
        const uint D = 1u << log_D;
        tLookupRange lookup(-(int)(1u << (log_len - 1)), 1u << log_len);
        FrTensor S(D), A(D);
        const std::unique_ptr<FrTensor> ints(new FrTensor(D / 8));
        const unsigned long before = fake_launched("carried_pair_kernelILi2E");          // the kind whose first round gathers
        try {
            lookup.prove(reinterpret_cast<const int*>(ints->gpu_data), S, A, random_vec(log_D), hyrax, cols, seconds);
        } catch (const std::exception&) {                    // nothing is computed here, so its claims do not hold
        }
        return fake_launched("carried_pair_kernelILi2E") - before;
    };
    expect(carried(8, 19) == 1 && carried(19, 19) == 1 && carried(24, 24) == 1, "tables of up to 2^24 entries");
    expect(carried(25, 25) == 0 && carried(30, 30) == 0, "longer ones are left to the weighted rounds");
    expect(carried(8, 18) == 0, "as are short proofs");
}

// A range of 2^23 entries has a row for each of them where rows are short (64 GiB for 64 columns): its indices, 2^23 among them, are
// digits of the widest radix there is.
static void the_longest_indexed_range() {
    const uint cols = 64, gens = 1u << 12, log_len = 23, D = 1u << log_len;
    bn128 G = bn128::one();
    Hyrax hyrax(1, gens, device_points(256 * (size_t)gens), G, 1);
    tLookupRange lookup(-(int)(D / 2), D);
    FrTensor S(D), A(D);
    const std::unique_ptr<FrTensor> ints(new FrTensor(D / 8));
    double seconds = 0;
    std::string error;
    const unsigned long before = fake_launched("scaled_chain");
    try {
        lookup.prove(reinterpret_cast<const int*>(ints->gpu_data), S, A, random_vec(log_len), hyrax, cols, seconds);
    } catch (const std::exception& e) {
        error = e.what();
    }
    expect(fake_launched("scaled_chain") > before, "the table is built");
    expect(error.find("tLookup_phase2: claim") == 0, "and the proof goes on to its claims, which do not hold here");
    uint32_t *out = reinterpret_cast<uint32_t*>(device_points(8)), *flag = reinterpret_cast<uint32_t*>(device_points(1));
    auto committed = [&](uint32_t len) {
        return grape_commit_indexed(out, reinterpret_cast<const int32_t*>(ints->gpu_data), 2 * cols, cols, out, cols, len, 0, nullptr, 0,
                                    reinterpret_cast<int32_t*>(flag), nullptr) == GRAPE_OK;
    };
    for (uint32_t len : {1u, 2u, 3u, 4u, 5u, 1u << 22, (1u << 23) - 1, 1u << 23}) expect(committed(len), "a table of that length");
    expect(!committed(0) && !committed((1u << 23) + 1), "none and more are refused");
}

// Rows start at the entry that witnesses are padded with where their table was made for a padded witness, or for a long one.
static void where_padding_is_free() {
    const uint cols = 64, gens = 1u << 12;
    bn128 G = bn128::one();
    Hyrax hyrax(1, gens, device_points(256 * (size_t)gens), G, 1);
    double seconds = 0;
    auto started = [&](tLookupRange& lookup, uint D) {
        const uint Dp = 1u << Log2(D);
        FrTensor S(Dp), A(Dp);
        S.set_size(D);
        const std::unique_ptr<FrTensor> ints(new FrTensor(D / 8));
        const unsigned long before = fake_launched("quad_affine_kernelILb1E");
        try {
            lookup.prove(reinterpret_cast<const int*>(ints->gpu_data), S, A, random_vec(Log2(D)), hyrax, cols, seconds);
        } catch (const std::exception&) {                    // nothing is computed here, so its claims do not hold
        }
        return fake_launched("quad_affine_kernelILb1E") - before;
    };
    tLookupRange even(-128, 256), padded(-128, 256), large(-128, 256);
    expect(started(even, 1u << 14) == 0 && started(even, 16 * 11008) == 0, "not for a short witness that is not padded");
    expect(started(padded, 16 * 11008) == 1 && started(padded, 1u << 14) == 1, "for one that is");
    expect(started(large, 1u << 20) == 1 && started(large, 16 * 11008) == 1, "for a long one");
}

// A mapping's witness is S_in + r S_out with the r its caller sees: read as T[index] while T was made with it, written out otherwise (the
// rounds then find that it is not T's).
static void a_mapping_with_another_r() {
    const uint cols = 64, log_D = 19, D = 1u << log_D;
    bn128 G = bn128::one();
    Hyrax hyrax(1, cols, device_points(256 * cols), G, 1);
    const std::vector<int> table(256, 7);
    tLookupRangeMapping lookup(-128, 256, table.data());
    double seconds = 0;
    auto written = [&] {
        FrTensor A(D);
        const std::unique_ptr<FrTensor> ints(new FrTensor(D / 8));
        const unsigned long before = fake_launched("index_embed_i32_kernel");
        const int* x = reinterpret_cast<const int*>(ints->gpu_data);
        try {
            lookup.prove(x, x, D, A, random_vec(log_D), hyrax, cols, seconds);
        } catch (const std::exception&) {                    // nothing is computed here, so its claims do not hold
        }
        return fake_launched("index_embed_i32_kernel") - before;
    };
    expect(written() == 0, "T's own r");
    const Fr own = lookup.r;
    lookup.r = own + Fr::one();
    expect(written() == 1, "another");
    lookup.r = own;
    expect(written() == 0, "T's own again");
}

// A lookup whose alpha is zero proves nothing about A (S + beta) = 1: its long rounds are refused, carried or not.  Nothing is computed
// here - every sum is zero - so the claim of such a proof holds and the refusal is the rule's.
static void lookups_without_a_weighted_term() {
    const uint cols = 64;
    bn128 G = bn128::one();
    Hyrax hyrax(1, cols, device_points(256 * cols), G, 1);
    double seconds = 0;
    auto refused = [&](uint log_D, Fr alpha) {
        const uint D = 1u << log_D;
        struct Lookup : tLookupRange {
            Lookup(const Fr& a) : tLookupRange(-128, 256) { alpha = a; }
        } lookup(alpha);
        FrTensor S(D), A(D);
        const std::unique_ptr<FrTensor> ints(new FrTensor(D / 8));
        try {
            lookup.prove(reinterpret_cast<const int*>(ints->gpu_data), S, A, random_vec(log_D), hyrax, cols, seconds);
        } catch (const std::exception& e) {
            return std::string(e.what()).find("a challenge is zero") != std::string::npos;
        }
        return false;
    };
    expect(refused(18, Fr::zero()), "two weighted long rounds");
    expect(refused(19, Fr::zero()) && refused(21, Fr::zero()), "carried ones");
    expect(!refused(10, Fr::zero()), "short rounds are all sums");
}

// The weights over the high variables are made for the proofs that read them: rounds of more than 2^20 weights and carried ones.
static void weights_that_are_read() {
    const uint cols = 64, len = 256;
    bn128 G = bn128::one();
    Hyrax hyrax(1, cols, device_points(256 * cols), G, 1);
    tLookupRange lookup(-128, len);
    double seconds = 0;
    auto pyramids = [&](uint log_D, bool ints) {
        const uint D = 1u << log_D;
        FrTensor S(D), A(D), S_out(D);
        int* x = reinterpret_cast<int*>(device_points(D / 16));
        const std::vector<int> map(len, 7);
        tLookupRangeMapping mapping(-128, len, map.data());
        const unsigned long before = fake_launched("eq_pyramid_head_kernel");
        try {
            if (ints) lookup.prove(x, S, A, random_vec(log_D), hyrax, cols, seconds);
            else mapping.prove(S, S_out, A, random_vec(log_D), hyrax, cols, seconds);
        } catch (const std::exception&) {
        }
        return fake_launched("eq_pyramid_head_kernel") - before;
    };
    expect(pyramids(16, true) == 1 && pyramids(17, true) == 1 && pyramids(18, true) == 1, "not for short proofs");
    expect(pyramids(19, true) == 2 && pyramids(22, true) == 2, "for carried weights");
    expect(pyramids(19, false) == 1 && pyramids(21, false) == 1 && pyramids(22, false) == 2, "without them, from 2^22 elements on");
}

// Mapping objects of the C calls are found by the mapped values: one other value is another object, also where the words it sits
// in agree under xor with a rotated product; the same values are the same object.
static void mapping_objects() {
    const uint32_t len = 1024, D = 2048, cols = 64;
    const uint32_t* ints = reinterpret_cast<uint32_t*>(device_points(64));
    const uint32_t* table = reinterpret_cast<uint32_t*>(device_points(256 * cols));
    uint32_t point[8 * 11] = {0}, alpha[8] = {1}, r[8] = {2}, transcript[32 * 16], rounds, claim[8];
    auto made = [&](const std::vector<int32_t>& map) {
        const unsigned long before = fake_launched("tl_table_kernel");          // the object's T
        grape_host_tlookup_mapping_prove(ints, ints, D, -512, len, map.data(), alpha, r, point, point, 11, table, cols, 1, cols, transcript, &rounds, claim);
        return fake_launched("tl_table_kernel") - before;
    };
    grape_host_set_input_format(1);
    std::vector<int32_t> map(len);
    for (uint32_t i = 0; i < len; i++) map[i] = (int32_t)(i * 2654435761u);
    const unsigned long first = made(map);
    expect(first > 0 && made(map) == 0, "the same values find their object");
    std::vector<int32_t> other(map);
    other[1] ^= INT32_MIN;
    other[16] ^= 1 << 26;
    expect(made(other) == first, "two changed words make another object");
    expect(made(map) == 0 && made(other) == 0, "both are kept");
    for (uint32_t i : {0u, 777u, len - 1}) {
        std::vector<int32_t> one(map);
        one[i] ^= 1;
        expect(made(one) == first, "one changed value makes another object");
    }
}

// Memory that a program gets is idle when it gets it, whatever was queued on it before: on the default stream, and - while the
// library itself has no further stream - on one it has never seen.  So the program may use it on a stream of its own at once.
static void tensor_memory_is_idle() {
    const uint n = 5000;
    FrTensor x(n);
    std::vector<Fr> host(n, Fr::one());
    int* ints = reinterpret_cast<int*>(device_points(n));
    const int unseen = 0;
    const std::map<std::string, std::function<std::shared_ptr<void>()>> sources = {
        {"a tensor", [&] { return std::make_shared<FrTensor>(n); }},
        {"a copy", [&] { return std::make_shared<FrTensor>(x); }},
        {"embedded integers", [&] { return std::make_shared<FrTensor>(n, ints); }},
        {"a tensor from the host", [&] { return std::make_shared<FrTensor>(FrTensor::from_host(host)); }},
        {"row sums", [&] { return std::make_shared<FrTensor>(x.sum(n, 1)); }},
        {"a vector of challenges", [&] { return std::shared_ptr<void>(grape_host::upload(host), [](void* p) { grape_free(p); }); }},
        {"a fold", [&] { return std::make_shared<FrTensor>(FrTensor::folded_from_ints(ints, n, x.gpu_data, 8, 0, n / 8)); }},
        {"a scalar", [&] { return std::make_shared<grape_host::DeviceFr>(host[0]); }},
    };
    for (const auto& s : sources) {
        s.second();                                          // leaves a block of that size behind
        grape_host::check(grape_stream_sync(nullptr), "sync");
        std::shared_ptr<void> first = s.second();
        grape_host::check(grape_memset_zero(x.gpu_data, 32, nullptr), "grape_memset_zero");     // stands for work on the block
        fake_queue(&unseen);
        const unsigned long on_default = fake_pending(nullptr);
        first.reset();
        const unsigned long before = fake_waits();
        const std::shared_ptr<void> second = s.second();
        expect(on_default > 0 && fake_waits() > before && fake_pending(&unseen) == 0, s.first.c_str());
    }
}

// The table that sparse commitments go through where rows hold many elements: not built for a short proof or two, built once
// such proofs have come up often enough, and never in the way of another table.
static void sparse_commitment_table() {
    const uint cols = 4096, D = 1u << 21;
    bn128 G = bn128::one();
    Hyrax hyrax(1, cols, device_points(256 * cols), G, 1);
    hyrax.set_table_budget((size_t)96 << 30);
    expect(hyrax.prepare_scaled_tables(cols), "the per-window table fits");
    FrTensor A(D);
    int* skip = reinterpret_cast<int*>(device_points(D / 16));
    auto prove = [&] { grape_free(hyrax.commit_sparse_affine(A, skip, D, cols, D / 2)); };
    const unsigned long start = fake_bytes();
    prove();
    prove();
    expect(fake_bytes() - start < (1ul << 30), "two short proofs build no table");
    for (int i = 0; i < 40; i++) prove();
    const unsigned long built = fake_bytes();
    expect(built - start > (8ul << 30), "forty do");
    FrTensor B(1u << 16);
    affine_t* scaled = hyrax.build_scaled_table(B, cols);
    expect(scaled != nullptr, "a lookup's table still fits");
    grape_free(hyrax.commit_affine(skip, 2 * cols, cols));
    expect(fake_bytes() - start > (47ul << 30), "and the one for 16-bit integers");
    Hyrax::release_scaled_table(scaled);
    // a table that a commitment of full rows finds in place stays
    Hyrax other(1, cols, hyrax.g_affine, G, 1);
    other.set_table_budget((size_t)96 << 30);
    expect(other.prepare_scaled_tables(cols), "the per-window table fits");
    for (int i = 0; i < 40; i++) grape_free(other.commit_sparse_affine(A, skip, D, cols, D / 2));
    grape_free(other.commit_affine(A, D, cols));
    expect(other.table_bytes_free() < (size_t)16 << 30 && other.build_scaled_table(B, cols) == nullptr, "a table in use by others does not give way");
}

// A scaled table that grows by moving: the budget holds the old and the new one, and where it or the device's memory does not, the
// table stays as it was.  One that there is no memory for is not made.
static void scaled_tables_that_grow() {
    const uint cols = 256, rows = 1u << 16;
    const unsigned long row_bytes = grape_g1_wide_table_bytes(cols, 1, 1);
    bn128 G = bn128::one();
    Hyrax hyrax(1, cols, device_points(256 * cols), G, 1);
    hyrax.set_table_budget((size_t)64 << 30);
    expect(hyrax.prepare_scaled_tables(cols), "the per-window table fits");
    FrTensor B(rows), more(1);
    affine_t* table = hyrax.build_scaled_table(B, cols);
    affine_t* const first = table;
    const size_t used = ((size_t)64 << 30) - hyrax.table_bytes_free();
    uint capacity = rows;
    auto unchanged = [&] { return table == first && capacity == rows && hyrax.table_bytes_free() + used <= (size_t)64 << 30; };
    // the eighth of the budget that tables may grow into holds the new one, the rest of it not the old one beside it
    FrTensor C((uint)((((size_t)64 << 30) - used - rows * row_bytes) / row_bytes));
    affine_t* rest = hyrax.build_scaled_table(C, cols);
    expect(table && rest && hyrax.table_bytes_free() > rows / 2 * row_bytes, "two tables, and room for half of the first");
    expect(!hyrax.extend_scaled_table(table, rows, capacity, more, cols) && unchanged(), "no room for both");
    Hyrax::release_scaled_table(rest);
    grape_host::check(grape_alloc_cache_release(nullptr), "grape_alloc_cache_release");
    fake_limit(fake_bytes() + (1ul << 30));
    expect(!hyrax.extend_scaled_table(table, rows, capacity, more, cols) && unchanged(), "no memory for both");
    expect(hyrax.build_scaled_table(B, cols) == nullptr && unchanged(), "none for another table");
    fake_limit(~0ul);
    expect(hyrax.extend_scaled_table(table, rows, capacity, more, cols) && table != first && capacity > rows, "with both it grows");
    const affine_t* second = table;
    expect(hyrax.extend_scaled_table(table, rows + 1, capacity, more, cols) && table == second, "and then in place");
    Hyrax::release_scaled_table(table);
}

// operands of the C calls at addresses that are multiples of 4 only
static void operands_at_any_address() {
    uint32_t* at = reinterpret_cast<uint32_t*>(device_points(4096));
    uint32_t point[8 * 16] = {0}, claim[8] = {0}, transcript[32 * 16], rounds, a[8], b[8];
    for (int shift = 0; shift < 4; shift++) {
        const uint32_t *A = at + shift, *B = at + 8 * 4096;
        expect(grape_host_prove_matmul(A, B, 1, 8, 8, 8, point, 6, point, 3, claim, transcript, &rounds, a, b) == 0, "matrix product, left");
        expect(grape_host_prove_matmul(B, A, 1, 8, 8, 8, point, 6, point, 3, claim, transcript, &rounds, a, b) == 0, "matrix product, right");
        expect(grape_host_prove_elemul(A, B, 1, 8, 8, point, 6, point, 6, claim, transcript, &rounds, a, b) == 0, "element product, left");
        expect(grape_host_prove_elemul(B, A, 1, 8, 8, point, 6, point, 6, claim, transcript, &rounds, a, b) == 0, "element product, right");
    }
}

// passes over the long rounds that carry their weights, two rounds each or one, and the launches that finish their sums
struct CarriedLaunches {
    unsigned long pairs = 0, singles = 0, finished = 0;
    static CarriedLaunches now() {
        CarriedLaunches c;
        c.pairs = fake_launched("carried_pair_kernel");
        c.singles = fake_launched("carried_round_kernel");
        c.finished = fake_launched("carried_final_kernel");
        return c;
    }
    CarriedLaunches since(const CarriedLaunches& before) const {
        CarriedLaunches c;
        c.pairs = pairs - before.pairs;
        c.singles = singles - before.singles;
        c.finished = finished - before.finished;
        return c;
    }
    unsigned long rounds() const { return 2 * pairs + singles; }
    bool none() const { return pairs + singles + finished == 0; }
    // every round but an odd one's last runs in a pass of two, and one launch finishes all sums
    bool carried(unsigned long n) const { return rounds() == n && singles == n % 2 && finished == 1; }
};

// An element product carries its weights where few rows are left in the end: each of them costs the host a factor.
static void element_products_that_carry() {
    uint32_t *a = reinterpret_cast<uint32_t*>(device_points(1u << 20)), claim[8] = {0}, transcript[32 * 32], rounds, at_a[8], at_b[8];
    std::vector<uint32_t> point(8 * 32, 3);
    auto product = [&](uint rows, uint cols) {
        const CarriedLaunches before = CarriedLaunches::now();
        const int vars = (int)Log2(rows) + (int)Log2(cols);
        grape_host_prove_elemul(a, a, 1, rows, cols, point.data(), vars, point.data(), vars, claim, transcript, &rounds, at_a, at_b);
        return CarriedLaunches::now().since(before);
    };
    grape_host_set_input_format(0);
    expect(product(1u << 10, 3000).carried(5) && product(1u << 11, 1u << 10).carried(5) && product(1u << 13, 257).carried(5), "from rows of 256 on");
    expect(product(1u << 11, 3000).carried(6), "an even number of rounds");
    expect(product(1u << 19, 5).none() && product(1u << 15, 65).none() && product(1u << 14, 255).none(), "not with shorter rows");
}

// A tensor times itself, both operands bound in the one buffer: the weighted half would overwrite the plain one, and from the second
// carried round on nothing compares them.  Two tensors of the same size carry.
static void a_tensor_times_itself() {
    const uint rows = 1u << 10, cols = 1u << 11;
    const std::vector<Fr> point(Log2(rows) + Log2(cols), Fr(3));
    auto product = [&](FrTensor& x, FrTensor& y) {
        const CarriedLaunches before = CarriedLaunches::now();
        Fr claim = Fr::zero();
        prove_eleMul(x, y, 1, rows, cols, point, point, claim);
        return CarriedLaunches::now().since(before);
    };
    FrTensor x(rows * cols), y(rows * cols);
    expect(product(x, y).carried(5), "two tensors carry");
    expect(product(x, x).none(), "one tensor does not");
}

// An opening that verifies here: every commitment is the identity (device memory reads as zero), so its two equations are
// commit_d == 0 and commit_ad == -(c * result) * G.
static Hyrax_proof trivial_opening(const bn128& G, const Fr& c, uint cols) {
    const Fr result(5);
    Hyrax_proof proof(result, cols, bn128::zero(), (Fr::zero() - c * result) * G);
    for (uint i = 0; i < cols; i++) proof.z[i] = Fr::zero();
    return proof;
}

// Openings of rows that are no power of two long: what the folds leave of integers, or a single row, is shorter than the padded row.
static void padded_openings() {
    const uint cols = 1100, gens = 2048;
    bn128 G = bn128::one();
    Hyrax hyrax(1, gens, device_points(256 * (size_t)gens), G, 1);
    const int* ints = reinterpret_cast<int*>(device_points(16 * cols));
    for (uint rows : {1u, 2u, 16u}) {
        FrTensor x(rows * cols);
        expect(hyrax.open(ints, random_vec(11 + Log2(rows)), Fr(3), rows * cols, cols).z_size == gens, "of integers");
        expect(hyrax.open(x, random_vec(11 + Log2(rows)), Fr(3), rows * cols, cols).z_size == gens, "of field elements");
    }
}

// a point with more variables than the rows need: the rows that are missing count as the identity
static void verify_with_more_variables() {
    const uint cols = 64, rows = 4;
    bn128 G = bn128::one();
    Hyrax hyrax(1, cols, device_points(256 * cols), G, 1);
    jacob_t* commitment = reinterpret_cast<jacob_t*>(device_points(2 * rows));
    const Fr c(3);
    Hyrax_proof proof = trivial_opening(G, c, cols);
    for (uint more : {0u, 1u, 20u, 40u}) {
        const unsigned long before = fake_bytes();
        expect(hyrax.verify(proof, commitment, random_vec(6 + 2 + more), c, rows * cols, cols), "the opening verifies");
        expect(fake_bytes() - before < (64ul << 20), "without a table over all variables");
    }
    Hyrax_proof wrong = trivial_opening(G + G, c, cols);
    expect(!hyrax.verify(wrong, commitment, random_vec(6 + 2 + 40), c, rows * cols, cols), "a wrong one does not");
}

// A check's single row goes without a table of its own where the device has no memory for it, and asks for it again only now and then.
static void single_rows_without_memory() {
    const uint cols = 4096, rows = 4;
    bn128 G = bn128::one();
    Hyrax hyrax(1, cols, device_points(256 * cols), G, 1);
    jacob_t* commitment = reinterpret_cast<jacob_t*>(device_points(2 * rows));
    const Fr c(3);
    Hyrax_proof proof = trivial_opening(G, c, cols);
    auto checked = [&] {
        const unsigned long before = fake_launched("wide_chain_kernel");
        expect(hyrax.verify(proof, commitment, random_vec(12 + 2), c, rows * cols, cols), "the opening verifies");
        return fake_launched("wide_chain_kernel") - before;
    };
    expect(checked() == 0, "the first row is worth no table");
    fake_limit(fake_bytes() + (64ul << 20));
    unsigned long tables = 0;
    for (int i = 0; i < 20; i++) tables += checked();
    expect(tables == 0, "without memory for one none is made");
    fake_limit(fake_bytes() + (3ul << 30));
    for (int i = 0; i < 20; i++) tables += checked();
    expect(tables == 1, "with it one");
    // rows of another length: there is memory for their table or for the one at hand, not for both
    Hyrax two(1, 2 * cols, device_points(256 * 2 * cols), G, 1);
    Hyrax_proof longer = trivial_opening(G, c, 2 * cols);
    auto check_two = [&](Hyrax_proof& p, uint n) { expect(two.verify(p, commitment, random_vec(Log2(n) + 2), c, rows * n, n), "the opening verifies"); };
    fake_limit(~0ul);
    for (int i = 0; i < 20; i++) check_two(proof, cols);
    const unsigned long at_hand = fake_launched("wide_chain_kernel");
    fake_limit(fake_bytes() + (1ul << 30));
    for (int i = 0; i < 20; i++) check_two(longer, 2 * cols);
    for (int i = 0; i < 20; i++) check_two(proof, cols);
    expect(at_hand == 2 && fake_launched("wide_chain_kernel") == at_hand, "the one at hand stays");
}

// The counter that a sum's workgroups take turns at is cleared before the first sum that uses it, also when the first attempt at that fails.
static void a_sum_behind_a_failed_one() {
    FrTensor x(4096);
    uint32_t *in = reinterpret_cast<uint32_t*>(x.gpu_data), *out = in + 8 * 2048;
    fake_fail_launches(1);
    expect(grape_fr_sum(out, in, 2000, nullptr) != GRAPE_OK, "the launch that clears it fails");
    const unsigned long cleared = fake_launched("zero_words_kernel"), sums = fake_launched("sum_kernelILb1E");
    expect(grape_fr_sum(out, in, 2000, nullptr) == GRAPE_OK && fake_launched("zero_words_kernel") == cleared + 1, "the next sum clears it");
    expect(grape_fr_sum(out, in, 2000, nullptr) == GRAPE_OK && fake_launched("zero_words_kernel") == cleared + 1, "the one behind it does not");
    expect(fake_launched("sum_kernelILb1E") == sums + 2, "both are sums in one launch");
}

// Which table a single row goes through: the reference-format one until such rows have cost a table, a strided one where there is one (its
// doublings count too), the row's own from then on.
static void tables_of_single_rows() {
    const uint cols = 512, rows = 4;
    bn128 G = bn128::one();
    jacob_t* commitment = reinterpret_cast<jacob_t*>(device_points(2 * rows));
    const Fr c(3);
    Hyrax_proof proof = trivial_opening(G, c, cols);
    auto path = [&](Hyrax& hyrax) {
        const unsigned long ref = fake_launched("commit_ref30_kernel"), strided = fake_launched("commit_strided_kernel"), wide = fake_launched("commit_wide_kernel");
        expect(hyrax.verify(proof, commitment, random_vec(9 + 2), c, rows * cols, cols), "the opening verifies");
        return std::string(fake_launched("commit_ref30_kernel") - ref, 'r') + std::string(fake_launched("commit_strided_kernel") - strided, 's') +
               std::string(fake_launched("commit_wide_kernel") - wide, 'w');
    };
    affine_t* gens = device_points(256 * cols);
    Hyrax first(1, cols, gens, G, 1), none(1, cols, gens, G, 1), second(1, cols, gens, G, 1);
    expect(path(first) == "r" && path(first) == "w" && path(first) == "w", "the reference-format table, then the row's own");
    none.set_table_budget(0);
    for (int i = 0; i < 5; i++) expect(path(none) == "r", "without a budget the reference-format table");
    // half of the budget for a strided table, the rest too little for the row's own
    second.set_table_budget((size_t)400 << 20);
    FrTensor two(2 * cols);
    grape_free(second.commit_affine(two, 2 * cols, cols));
    expect(path(second) == "s", "a strided table");
    for (int i = 0; i < 20; i++) expect(path(second) == "s", "for good where the row's own does not fit beside it");
}

// The table for single rows is in no other table's way: it goes for one that needs its bytes, and for a per-window table that serves
// its rows, and it is not made where a table that gives way itself would have to go for it.
static void single_row_table_gives_way() {
    const uint cols = 4096, rows = 4;
    bn128 G = bn128::one();
    affine_t* gens = device_points(256 * cols);
    jacob_t* commitment = reinterpret_cast<jacob_t*>(device_points(2 * rows));
    const Fr c(3);
    Hyrax_proof proof = trivial_opening(G, c, cols);
    auto check_rows = [&](Hyrax& hyrax) {
        const unsigned long before = fake_launched("wide_chain_kernel");
        for (int i = 0; i < 20; i++) expect(hyrax.verify(proof, commitment, random_vec(12 + 2), c, rows * cols, cols), "the opening verifies");
        return fake_launched("wide_chain_kernel") - before;
    };
    int* ints = reinterpret_cast<int*>(device_points(4 * cols));
    {
        Hyrax hyrax(1, cols, gens, G, 1);
        hyrax.set_table_budget((size_t)16 << 30);
        expect(check_rows(hyrax) == 1, "single rows have a table");
        const unsigned long before = fake_bytes();
        grape_free(hyrax.commit_affine(ints, 2 * cols, cols));
        expect(fake_bytes() - before > (13ul << 30), "the one for 16-bit integers takes its place");
        expect(check_rows(hyrax) == 0, "and keeps it");
    }
    {
        Hyrax hyrax(1, cols, gens, G, 1), other(1, cols, gens, G, 1);
        expect(check_rows(hyrax) == 1 && other.prepare_scaled_tables(cols), "single rows have a table");
        grape_host::check(grape_alloc_cache_release(nullptr), "grape_alloc_cache_release");
        const unsigned long before = fake_bytes();
        expect(hyrax.prepare_scaled_tables(cols), "the per-window table fits");
        grape_host::check(grape_alloc_cache_release(nullptr), "grape_alloc_cache_release");
        expect(fake_bytes() - before < grape_g1_wide_table_bytes(cols, 20, 1u << 12) - (1ul << 30), "and serves them too");
        expect(check_rows(hyrax) == 0, "so that no other is made");
    }
    Hyrax hyrax(1, cols, gens, G, 1);
    hyrax.set_table_budget((size_t)96 << 30);
    FrTensor A(1u << 21);
    int* skip = reinterpret_cast<int*>(device_points(1u << 17));
    const unsigned long none = fake_bytes();
    for (int i = 0; i < 40; i++) grape_free(hyrax.commit_sparse_affine(A, skip, A.size, cols, A.size / 2));
    const unsigned long spare = fake_bytes() - none;
    expect(spare > (8ul << 30), "sparse commitments have a table");
    hyrax.set_table_budget(spare + (1ul << 30));
    const unsigned long before = fake_bytes();
    expect(check_rows(hyrax) == 0 && fake_bytes() >= before, "single rows do not take its place");
}

// the generator of an object is replaced between two checks
static void verify_with_another_generator() {
    const uint cols = 64, rows = 4;
    bn128 G = bn128::one();
    Hyrax hyrax(1, cols, device_points(256 * cols), G, 1);
    jacob_t* commitment = reinterpret_cast<jacob_t*>(device_points(2 * rows));
    const Fr c(3);
    const std::vector<Fr> point = random_vec(8);
    Hyrax_proof first = trivial_opening(G, c, cols), second = trivial_opening(G + G, c, cols);
    expect(hyrax.verify(first, commitment, point, c, rows * cols, cols), "the opening verifies");
    hyrax.G = G + G;
    expect(!hyrax.verify(first, commitment, point, c, rows * cols, cols), "an opening under the old generator does not verify under the new one");
    expect(hyrax.verify(second, commitment, point, c, rows * cols, cols), "one under the new generator does");
}

// A short copy from a block that belongs to another device than the thread's current one goes through the runtime, which reads it
// there: no kernel of this device does.  And a kept block is not handed out on another device.
static void blocks_of_two_devices() {
    void *p = nullptr, *q = nullptr;
    grape_host::ensure_init();
    grape_host::check(grape_malloc(&p, 1 << 21), "grape_malloc");
    char out[256];
    const unsigned long launches = fake_launches(), copies = fake_copies();
    grape_host::check(grape_memcpy_d2h(out, p, sizeof out, nullptr), "grape_memcpy_d2h");
    expect(fake_launches() == launches + 1 && fake_copies() == copies, "a kernel reads a block of the current device");
    fake_set_device(1);
    grape_host::check(grape_memcpy_d2h(out, p, sizeof out, nullptr), "grape_memcpy_d2h");
    expect(fake_launches() == launches + 1 && fake_copies() == copies + 1, "the runtime copies from another device");
    grape_host::check(grape_free(p), "grape_free");
    grape_host::check(grape_malloc(&q, 1 << 21), "grape_malloc");
    expect(q != p, "a block stays with its device");
    fake_set_device(0);
    grape_host::check(grape_malloc(&q, 1 << 21), "grape_malloc");
    expect(q == p, "and is handed out there");
}

// Blocks that only the default stream works on: handed on with no wait while every other stream is one the library joins itself;
// waited for when a caller's stream is about, and when memory for any stream takes them over.
static void default_order_blocks() {
    auto get = [](bool on_default) {
        void* p = nullptr;
        grape_host::check((on_default ? grape_malloc_on_default : grape_malloc)(&p, 5000), "grape_malloc");
        return p;
    };
    grape_host::ensure_init();
    grape_stream_t side, user;
    grape_host::check(grape_stream_create(&side), "grape_stream_create");
    grape_host::check(grape_stream_internal(side), "grape_stream_internal");
    auto work = [](void* p, grape_stream_t st) { grape_host::check(grape_memset_zero(p, 64, st), "grape_memset_zero"); };
    void* p = get(true);
    work(p, nullptr);
    grape_host::check(grape_free_on_default(p), "grape_free");
    unsigned long waits = fake_waits();
    void* q = get(true);
    expect(q == p && fake_waits() == waits && fake_pending(nullptr) == 1, "handed on in the default stream's order");
    grape_host::check(grape_free_on_default(q), "grape_free");
    q = get(false);
    expect(q == p && fake_pending(nullptr) == 0, "memory for any stream waits for the default stream");
    work(q, side);
    grape_host::check(grape_free(q), "grape_free");
    q = get(true);
    expect(q == p && fake_pending(side) == 0, "a block of another kind is waited for");
    grape_host::check(grape_stream_create(&user), "grape_stream_create");
    work(q, user);
    grape_host::check(grape_free_on_default(q), "grape_free");
    q = get(true);
    expect(q == p && fake_pending(user) == 0, "a caller's stream is waited for");
    grape_host::check(grape_free_on_default(q), "grape_free");
    grape_host::check(grape_stream_destroy(user), "grape_stream_destroy");
    q = get(true);
    work(q, nullptr);
    grape_host::check(grape_free_on_default(q), "grape_free");
    waits = fake_waits();
    q = get(true);
    expect(q == p && fake_waits() == waits, "until it is gone");
    work(q, reinterpret_cast<grape_stream_t>(&waits));       // a stream that the caller brings
    grape_host::check(grape_free_on_default(q), "grape_free");
    q = get(true);
    expect(q == p && fake_pending(&waits) == 0, "a stream that a caller brings is waited for");
}

// A short copy goes through the kernel where it lies inside one block, through the runtime where it does not.
static void short_copies() {
    const size_t bytes = 1 << 20;
    char *p = nullptr, out[512];
    grape_host::ensure_init();
    grape_host::check(grape_malloc((void**)&p, bytes), "grape_malloc");
    auto by_kernel = [&](const void* from, size_t n) {
        const unsigned long launches = fake_launches(), copies = fake_copies();
        grape_host::check(grape_memcpy_d2h(out, from, n, nullptr), "grape_memcpy_d2h");
        expect(fake_launches() + fake_copies() == launches + copies + 1, "one launch or one copy");
        return fake_launches() > launches;
    };
    expect(by_kernel(p, 256) && by_kernel(p + bytes - 256, 256), "the first and the last bytes of a block");
    expect(!by_kernel(p + bytes - 252, 256) && !by_kernel(p + bytes - 4, 8), "a range that ends behind its block");
    expect(!by_kernel(p + 2, 4) && !by_kernel(p, 3), "addresses and lengths that are no words");
    expect(!by_kernel(out, 4), "host memory");
    grape_host::check(grape_free(p), "grape_free");
}

int main(int argc, char** argv) {
    const std::map<std::string, std::function<void()>> scenarios = {
        {"refused_lookup", refused_lookup},
        {"proof_after_a_refused_one", proof_after_a_refused_one},
        {"mapping_objects", mapping_objects},
        {"carried_lookups", carried_lookups},
        {"the_longest_indexed_range", the_longest_indexed_range},
        {"where_padding_is_free", where_padding_is_free},
        {"a_mapping_with_another_r", a_mapping_with_another_r},
        {"lookups_without_a_weighted_term", lookups_without_a_weighted_term},
        {"weights_that_are_read", weights_that_are_read},
        {"tensor_memory_is_idle", tensor_memory_is_idle},
        {"sparse_commitment_table", sparse_commitment_table},
        {"scaled_tables_that_grow", scaled_tables_that_grow},
        {"operands_at_any_address", operands_at_any_address},
        {"element_products_that_carry", element_products_that_carry},
        {"a_tensor_times_itself", a_tensor_times_itself},
        {"padded_openings", padded_openings},
        {"verify_with_more_variables", verify_with_more_variables},
        {"single_rows_without_memory", single_rows_without_memory},
        {"a_sum_behind_a_failed_one", a_sum_behind_a_failed_one},
        {"tables_of_single_rows", tables_of_single_rows},
        {"single_row_table_gives_way", single_row_table_gives_way},
        {"verify_with_another_generator", verify_with_another_generator},
        {"blocks_of_two_devices", blocks_of_two_devices},
        {"default_order_blocks", default_order_blocks},
        {"short_copies", short_copies},
    };
    auto it = scenarios.find(argc > 1 ? argv[1] : "");
    if (it == scenarios.end()) return 2;
    try {
        it->second();
    } catch (const std::exception& e) {
        std::printf("%s\n", e.what());
        return 1;
    }
    return failures ? 1 : 0;
}
