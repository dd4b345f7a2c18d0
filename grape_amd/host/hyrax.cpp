#include "hyrax.hpp"
#include <cstdlib>
#include <algorithm>
#include <cassert>
#include <cstring>
#include <map>
#include <utility>
#include "../../include/grape_hip.h"

using grape_host::check;
using grape_host::OnDefaultStream;
static inline uint32_t* W(void* p) { return reinterpret_cast<uint32_t*>(p); }
static inline const uint32_t* W(const void* p) { return reinterpret_cast<const uint32_t*>(p); }

Hyrax_proof::Hyrax_proof(Fr result_, size_t z_len, bn128 commit_d_, bn128 commit_ad_)
    : z_size(z_len), result(result_), commit_d(commit_d_), commit_ad(commit_ad_) {
    z = new Fr[z_size];
}
Hyrax_proof::~Hyrax_proof() { delete[] z; }
Hyrax_proof::Hyrax_proof(const Hyrax_proof& o) : z_size(o.z_size), result(o.result), commit_d(o.commit_d), commit_ad(o.commit_ad) {
    z = new Fr[z_size];
    for (size_t i = 0; i < z_size; i++) z[i] = o.z[i];
}
Hyrax_proof& Hyrax_proof::operator=(const Hyrax_proof& o) {
    if (this != &o) {
        delete[] z;
        z_size = o.z_size;
        result = o.result;
        commit_d = o.commit_d;
        commit_ad = o.commit_ad;
        z = new Fr[z_size];
        for (size_t i = 0; i < z_size; i++) z[i] = o.z[i];
    }
    return *this;
}

Hyrax::Hyrax(uint layer_num_, uint npoints_, affine_t* g, bn128& G_, uint com_scale_)
    : com_scale(com_scale_), layer_num(layer_num_), npoints(npoints_ * com_scale_), G(G_), g_affine(g) {
    grape_host::ensure_init();
    // GRAPE_TABLE_BUDGET_GIB overrides the default budget of the fixed-base tables
    if (const char* e = std::getenv("GRAPE_TABLE_BUDGET_GIB")) {
        char* end = nullptr;
        unsigned long long gib = std::strtoull(e, &end, 10);
        if (end != e) table_budget_ = (size_t)gib << 30;
    }
}
// scaled tables handed out: table -> the Hyrax object whose budget holds it, its bytes, whether it has been extended.  Never
// destroyed: lookup objects with static lifetime release their tables while the process exits.
namespace {
struct ScaledTable {
    Hyrax* owner = nullptr;
    size_t bytes = 0;
    bool extended = false;
};
}  // namespace
static std::map<const void*, ScaledTable>& scaled_registry() {
    static auto* r = new std::map<const void*, ScaledTable>();
    return *r;
}

Hyrax::~Hyrax() {
    for (auto& e : scaled_registry())
        if (e.second.owner == this) e.second.owner = nullptr;
    grape_free(int16_table_.d);
    grape_free(int16x2_table_.d);
    grape_free(int32_table_.d);
    grape_free(fr_table_.d);
    grape_free(row_table_.d);
    grape_free(fr_strided_.d);
}

// src/Hyrax.cu:314-315 / :337-338
void Hyrax::check_shape(uint size, uint N) const {
    if (size / N / com_scale < layer_num) throw std::runtime_error("Size too small: size < N * com_scale * layer_num");
    if (N != (1u << Log2(N))) throw std::runtime_error("N must be a power of 2");
}

// Builds (once) the wide table over the first `rowlen` generators; false when it exceeds the budget.  `optional`: also when there is no
// device memory for it beside the one it would replace, which then stays.
bool Hyrax::ensure_table(WideTable& t, uint rowlen, uint c, uint nw, uint K, bool optional) {
    if (t.d && t.ngen >= rowlen && t.c == c && t.nw == nw) return true;
    size_t bytes = grape_g1_wide_table_bytes(rowlen, nw, K);
    // against what every other table of this object holds (the one being replaced gives its bytes back)
    if (optional) {
        // none of the others goes for it, and the one it would replace is there until it is made
        if (table_bytes_in_use() + (fr_strided_.spare ? strided_bytes() : 0) + bytes_of(t) + bytes > table_budget_) return false;
    } else if (!make_room(bytes, bytes_of(t))) {
        return false;
    }
    if (rowlen > npoints) throw std::runtime_error("row longer than the generator set");
    if (!optional) {
        grape_free(t.d);
        t = WideTable();
    }
    affine_t* d = nullptr;
    int rc = grape_malloc((void**)&d, bytes);
    // generators are row k = 1 of the reference-format table
    if (rc == GRAPE_OK) rc = grape_g1_wide_table_gen(W(d), W(g_affine + npoints), rowlen, c, nw, K, nullptr);
    if (rc != GRAPE_OK) {
        grape_free(d);
        if (optional && rc == GRAPE_ENOMEM) return false;
        check(rc, "a table over the generators");
    }
    grape_free(t.d);
    t.d = d;
    t.ngen = rowlen;
    t.c = c;
    t.nw = nw;
    t.K = K;
    return true;
}

namespace {
// One C-ABI commitment call takes at most 2^28 scalars (the largest single call that is tested on the
// GPU); longer tensors go through in whole rows, each call writing its own rows of the output.
constexpr size_t kMaxScalarsPerCall = (size_t)1 << 28;
// fn(first_element, elements, first_row) -> status; stops at the first non-zero status
template <class F>
int for_row_chunks(size_t size, uint rowlen, F fn) {
    size_t rows_per_call = kMaxScalarsPerCall / rowlen;
    if (rows_per_call < 1) rows_per_call = 1;
    const size_t rows = size / rowlen;
    for (size_t r0 = 0; r0 < rows; r0 += rows_per_call) {
        const size_t nr = rows - r0 < rows_per_call ? rows - r0 : rows_per_call;
        int rc = fn(r0 * rowlen, nr * rowlen, r0);
        if (rc != GRAPE_OK) return rc;
    }
    return GRAPE_OK;
}
}  // namespace

affine_t* Hyrax::commit_affine(int* tensor, uint size, uint N) {
    check_shape(size, N);
    const uint rowlen = N * com_scale;
    const uint rows = size / rowlen;
    affine_t* out = nullptr;
    check(grape_malloc((void**)&out, sizeof(affine_t) * (size_t)rows), "grape_malloc");
    // small-scalar fast paths: one signed 16-bit digit per scalar (one mixed addition per element)
    // when that table fits the budget, else two signed 9-bit digits (two additions; 17 GB instead of
    // 275 GB for the 262144-column rows of the reference's com_scale = 16 shapes)
    if (int16_ok_) {
        WideTable* t = nullptr;
        if (ensure_table(int16_table_, rowlen, 16, 1, 32768)) t = &int16_table_;
        else if (ensure_table(int16x2_table_, rowlen, 9, 2, 256)) t = &int16x2_table_;
        if (t) {
            int rc = for_row_chunks(size, rowlen, [&](size_t e0, size_t n, size_t r0) {
                return grape_commit_i32(W(out + r0), tensor + e0, n, rowlen, W(t->d), t->ngen, t->c, t->nw, t->K, nullptr);
            });
            if (rc == GRAPE_OK) return out;
            if (rc != GRAPE_EINVAL) check(rc, "grape_commit_i32");
            int16_ok_ = false;   // a scalar outside int16: use the general tables from now on
        }
    }
    commit_i32_rows(out, tensor, size, rowlen, nullptr);
    return out;
}

// any int32 scalars: five signed 8-bit digits per scalar through a small table, or the reference's
// byte windows when even that table is over budget
void Hyrax::commit_i32_rows(affine_t* out, int* tensor, size_t size, uint rowlen, int* d_flag, void* stream) {
    if (!d_flag) stream = nullptr;                       // a call that waits for its result runs on the default stream
    const affine_t* had = int32_table_.d;
    if (ensure_table(int32_table_, rowlen, 8, 5, 128)) {
        // a table built just now was built on the default stream: another stream may read it only once it is there
        if (stream && int32_table_.d != had) check(grape_stream_sync(nullptr), "sync");
        check(for_row_chunks(size, rowlen, [&](size_t e0, size_t n, size_t r0) {
                  if (d_flag)
                      return grape_commit_i32_nowait(W(out + r0), tensor + e0, n, rowlen, W(int32_table_.d), int32_table_.ngen, 8, 5, 128,
                                                     d_flag, stream);
                  return grape_commit_i32(W(out + r0), tensor + e0, n, rowlen, W(int32_table_.d), int32_table_.ngen, 8, 5, 128, nullptr);
              }),
              "grape_commit_i32");
    } else {
        check(for_row_chunks(size, rowlen, [&](size_t e0, size_t n, size_t r0) {
                  return grape_commit_i32_ref_table(W(out + r0), tensor + e0, n, rowlen, W(g_affine), npoints, stream);
              }),
              "grape_commit_i32_ref_table");
    }
}

affine_t* Hyrax::commit_affine_i32(int* tensor, uint size, uint N, int* d_flag, void* stream) {
    check_shape(size, N);
    const uint rowlen = N * com_scale;
    affine_t* out = nullptr;
    check(grape_malloc((void**)&out, sizeof(affine_t) * (size_t)(size / rowlen)), "grape_malloc");
    commit_i32_rows(out, tensor, size, rowlen, d_flag, stream);
    return out;
}

size_t Hyrax::strided_bytes() const {
    return fr_strided_.d ? grape_g1_wide_table_bytes(fr_strided_.ngen, fr_strided_.nsets, 1u << (fr_strided_.c - 1)) : 0;
}
size_t Hyrax::bytes_of(const WideTable& t) { return t.d ? grape_g1_wide_table_bytes(t.ngen, t.nw, t.K) : 0; }
// without the tables that give way (make_room)
size_t Hyrax::table_bytes_in_use() const {
    size_t used = scaled_bytes_;
    for (const WideTable* t : {&int16_table_, &int16x2_table_, &int32_table_, &fr_table_}) used += bytes_of(*t);
    return fr_strided_.spare ? used : used + strided_bytes();
}
void Hyrax::drop_row_table() {
    grape_free(row_table_.d);
    row_table_ = WideTable();
}
// Is there room in the budget for a table of `bytes` that replaces one of `replaced` bytes?  Two tables go if they stand in the way:
// first the one for single rows, which saves a row a millisecond at most, then a strided table that only sparse
// commitments asked for: it saves them a fifth to a half of their additions, while a scaled or int16
// table that is not there costs 16 additions instead of one, or 2.
bool Hyrax::make_room(size_t bytes, size_t replaced) {
    const size_t used = table_bytes_in_use() - replaced;
    if (used + bytes > table_budget_) return false;
    const size_t spare = fr_strided_.spare ? strided_bytes() : 0;
    if (used + spare + bytes_of(row_table_) + bytes > table_budget_) drop_row_table();
    if (spare && used + spare + bytes > table_budget_) {
        grape_free(fr_strided_.d);
        fr_strided_ = StridedTable();
    }
    return true;
}

// A per-window table for full-width scalars (every window has its own set of multiples, so a
// scalar multiple needs additions only and one accumulator per lane): what the scaled table
// B[t] * G_i of a lookup object is built through and what the sparse commitment reads, at one
// addition per window (c = 13: 20 additions from 43 GB for 4096 generators; the widest window whose
// table stays below its cap and inside the budget is taken - the table itself is generated in a
// tenth of a second).  Multi-row commitments do not use it when a strided table exists.
bool Hyrax::ensure_fr_table(uint rowlen, bool build) {
    if (fr_table_.d && fr_table_.ngen >= rowlen) return true;
    if (!build) return false;
    const size_t used = table_bytes_in_use();
    for (uint c = 13; c >= 8; c--) {
        const uint nw = (255 + c - 1) / c, K = 1u << (c - 1);
        const size_t bytes = grape_g1_wide_table_bytes(rowlen, nw, K);
        // wide windows may take 48 GB, narrow ones (which lose to the strided table anyway) 16 GB
        const size_t cap = (size_t)(c >= 12 ? 48 : 16) << 30;
        if (bytes <= cap && used + bytes <= table_budget_) {
            if (!ensure_table(fr_table_, rowlen, c, nw, K)) return false;
            if (row_table_.ngen <= fr_table_.ngen) drop_row_table();     // single rows go through this one now
            return true;
        }
    }
    return false;
}

// Full-width scalars cost one addition per c-bit window, so the table that leaves the fewest
// additions per scalar within its share of the budget is built: windows of c bits, every J-th
// window set kept, the J residue sums combined by (J-1)*c doublings per row.  Measured cost per
// scalar, in additions: ceil(255/c) + 0.3 J (each residue recodes the scalar again).  Half of the
// budget at most goes to this table - the rest is for the int16 table and the lookups' scaled
// tables.  4096 generators: c = 16, J = 4, 4 sets, 69 GB, 16 additions (a per-window table of the
// same bytes has c = 14 and 19); 65536 generators: c = 13, J = 10; 262144: c = 11, J = 12, against
// 32 additions plus a doubling chain per row for the reference's byte windows.
// With worth_ms it is built where that takes no longer than worth_ms, and marked as a table that gives way to others; once
// a call that builds at any price has found it in place it stays.
bool Hyrax::ensure_strided_table(uint rowlen, bool build, const double* worth_ms) {
    if (fr_strided_.d && fr_strided_.ngen >= rowlen) {
        if (build && !worth_ms) fr_strided_.spare = false;
        return true;
    }
    if (!build) return false;
    if (rowlen > npoints) throw std::runtime_error("row longer than the generator set");
    const size_t used = table_bytes_in_use() - (fr_strided_.spare ? 0 : strided_bytes());
    size_t cap = table_budget_ / 2;
    if (used + cap > table_budget_) cap = table_budget_ > used ? table_budget_ - used : 0;
    // the cheapest table over `ngen` generators within the cap: cost per scalar, c, J, number of sets
    struct Choice { double cost; uint c, J, nsets; };
    auto choose = [&](uint ngen) {
        Choice best{30.0, 0, 0, 0};       // a table that does not beat 30 additions per scalar is not worth building
        for (uint c = 8; c <= 17; c++) {
            const uint nw = (255 + c - 1) / c;
            for (uint J = 1; J <= nw; J++) {
                const uint nsets = (nw + J - 1) / J;
                if ((nsets - 1) * J * c >= 256) continue;
                const size_t bytes = grape_g1_wide_table_bytes(ngen, nsets, 1u << (c - 1));
                if (bytes > cap) continue;
                const double cost = nw + 0.3 * J + (double)bytes / 1e12;
                if (cost < best.cost) best = Choice{cost, c, J, nsets};
            }
        }
        return best;
    };
    // one table over every generator serves all row lengths; it is preferred to a table over the
    // first `rowlen` generators (which a longer row would have to replace, at a tenth of a second per
    // build) unless that costs over a quarter more additions per scalar
    Choice pick = choose(rowlen);
    uint ngen = rowlen;
    if (npoints > rowlen) {
        const Choice all = choose(npoints);
        if (all.c != 0 && (pick.c == 0 || all.cost <= 1.25 * pick.cost)) {
            pick = all;
            ngen = npoints;
        }
    }
    const uint bc = pick.c, bj = pick.J, bs = pick.nsets;
    if (bc == 0) return false;
    // 64 GiB in 92 ms, 48 in 72 (4096 generators)
    const double build_ms = 1.35e-9 * (double)grape_g1_wide_table_bytes(ngen, bs, 1u << (bc - 1));
    if (worth_ms && (build_ms > *worth_ms || (fr_strided_.d && !fr_strided_.spare))) return false;
    if (used + grape_g1_wide_table_bytes(ngen, bs, 1u << (bc - 1)) + bytes_of(row_table_) > table_budget_) drop_row_table();
    grape_free(fr_strided_.d);
    fr_strided_ = StridedTable();
    check(grape_malloc((void**)&fr_strided_.d, grape_g1_wide_table_bytes(ngen, bs, 1u << (bc - 1))), "grape_malloc");
    check(grape_g1_strided_table_gen(W(fr_strided_.d), W(g_affine + npoints), ngen, bc, bj, bs, nullptr), "grape_g1_strided_table_gen");
    fr_strided_.ngen = ngen;
    fr_strided_.c = bc;
    fr_strided_.J = bj;
    fr_strided_.nsets = bs;
    fr_strided_.spare = worth_ms != nullptr;
    return true;
}

// A single row (an opening's blinding row, the z of its check) is a short accumulation and a chain: through a per-window table, which
// leaves no doublings, where there is one.  A strided table leaves (J - 1) c of them and the reference-format table 248, one
// after the other on four lanes, 4.5 us each (4096 columns, whole openings: 0.4 and 1.5 ms against 0.3).  So for the first row behind
// those that have spent on doublings what a small table takes to make - 8-bit windows, 2 GiB and 3 ms for 4096 generators - it is
// made; wider rows than 8192 would take more memory than an opening is worth.  It gives way to any other table, and to the per-window one
// over as many generators for good.
const Hyrax::WideTable* Hyrax::single_row_table(uint rowlen, void* stream) {
    if (ensure_fr_table(rowlen, false)) return &fr_table_;
    constexpr uint c = 8, nw = 32, K = 128;
    if (row_table_.d && row_table_.ngen >= rowlen) return &row_table_;
    const size_t bytes = grape_g1_wide_table_bytes(rowlen, nw, K);
    if (rowlen > npoints || bytes > (size_t)4 << 30) return nullptr;
    if (row_saving_ms_ < 0.2 + 1.35e-9 * (double)bytes) {
        const bool strided = fr_strided_.d && fr_strided_.ngen >= rowlen;
        row_saving_ms_ += 4.5e-3 * (strided ? (fr_strided_.J - 1) * fr_strided_.c : 248);
        return nullptr;
    }
    row_saving_ms_ = 0;                                         // where there is no memory for it: tried again after as much
    if (!ensure_table(row_table_, rowlen, c, nw, K, true)) return nullptr;
    if (stream) check(grape_stream_sync(nullptr), "sync");      // made on the default stream: another may read it only once it is there
    return &row_table_;
}

bool Hyrax::commit_fr_rows(affine_t* out, fr_t* scalars, size_t size, uint rowlen, bool may_build, void* stream, int* d_flag) {
    const WideTable* own = size == rowlen ? single_row_table(rowlen, stream) : nullptr;
    if (own) {
        const WideTable& t = *own;
        if (d_flag) {
            check(grape_commit_fr_nowait(W(out), W(scalars), size, rowlen, W(t.d), t.ngen, t.c, t.nw, t.K, d_flag, stream), "grape_commit_fr_nowait");
            return true;
        }
        check(grape_commit_fr(W(out), W(scalars), size, rowlen, W(t.d), t.ngen, t.c, t.nw, t.K, stream), "grape_commit_fr");
    } else if (ensure_strided_table(rowlen, may_build)) {
        const StridedTable& t = fr_strided_;
        check(for_row_chunks(size, rowlen, [&](size_t e0, size_t n, size_t r0) {
                  return grape_commit_fr_strided(W(out + r0), W(scalars + e0), n, rowlen, W(t.d), t.ngen, t.c, t.J, t.nsets, stream);
              }),
              "grape_commit_fr_strided");
    } else if (ensure_fr_table(rowlen, false)) {
        const WideTable& t = fr_table_;
        check(for_row_chunks(size, rowlen, [&](size_t e0, size_t n, size_t r0) {
                  return grape_commit_fr(W(out + r0), W(scalars + e0), n, rowlen, W(t.d), t.ngen, t.c, t.nw, t.K, stream);
              }),
              "grape_commit_fr");
    } else {
        check(for_row_chunks(size, rowlen, [&](size_t e0, size_t n, size_t r0) {
                  return grape_commit_fr_ref_table(W(out + r0), W(scalars + e0), n, rowlen, W(g_affine), npoints, stream);
              }),
              "grape_commit_fr_ref_table");
    }
    return false;
}

affine_t* Hyrax::commit_affine(FrTensor& tensor, uint size, uint N) {
    check_shape(size, N);
    const uint rowlen = N * com_scale;
    const uint rows = size / rowlen;
    affine_t* out = nullptr;
    check(grape_malloc((void**)&out, sizeof(affine_t) * (size_t)rows), "grape_malloc");
    commit_fr_rows(out, tensor.gpu_data, size, rowlen, rows > 1);
    return out;
}

affine_t* Hyrax::commit_row(FrTensor& row) {
    if (row.size > npoints) throw std::runtime_error("row longer than the generator set");
    affine_t* out = nullptr;
    check(grape_malloc((void**)&out, sizeof(affine_t)), "grape_malloc");
    commit_fr_rows(out, row.gpu_data, row.size, row.size, false);
    return out;
}

bool Hyrax::prepare_scaled_tables(uint ncols) { return ensure_fr_table(ncols); }

affine_t* Hyrax::build_scaled_table(const FrTensor& scalars, uint ncols) {
    if (ncols > npoints) throw std::runtime_error("row longer than the generator set");
    size_t bytes = grape_g1_wide_table_bytes(ncols, 1, scalars.size);   // one entry per (scalar, column)
    if (table_bytes_in_use() + bytes > table_budget_) return nullptr;      // before the per-window table is built for nothing
    if (!ensure_fr_table(ncols)) return nullptr;
    if (!make_room(bytes, 0)) return nullptr;
    affine_t* out = nullptr;
    int rc = grape_malloc((void**)&out, bytes);
    if (rc == GRAPE_OK) rc = gen_scaled(out, scalars, ncols);
    if (rc != GRAPE_OK) {
        grape_free(out);
        if (rc == GRAPE_ENOMEM) return nullptr;
        check(rc, "a scaled table");
    }
    scaled_bytes_ += bytes;
    scaled_registry()[out] = ScaledTable{this, bytes, false};
    return out;
}

int Hyrax::gen_scaled(affine_t* out, const FrTensor& scalars, uint ncols) {
    return grape_g1_scaled_table_gen(W(out), W(scalars.gpu_data), scalars.size, ncols, W(fr_table_.d), fr_table_.ngen, fr_table_.c, fr_table_.nw,
                                     fr_table_.K, nullptr);
}

size_t Hyrax::most_scaled_rows(const affine_t* table, uint ncols) const {
    size_t share = table_budget_ / 8;
    for (const auto& e : scaled_registry())
        if (e.second.owner == this && e.second.extended && e.first != table) share -= std::min(share, e.second.bytes);
    return share / grape_g1_wide_table_bytes(ncols, 1, 1);
}

bool Hyrax::extend_scaled_table(affine_t*& table, uint rows, uint& capacity, const FrTensor& more, uint ncols) {
    auto it = scaled_registry().find(table);
    if (it == scaled_registry().end() || it->second.owner != this) return false;
    const size_t row_bytes = grape_g1_wide_table_bytes(ncols, 1, 1), need = (size_t)rows + more.size, most = most_scaled_rows(table, ncols);
    if (need > most || !ensure_fr_table(ncols)) return false;
    if (need > capacity) {
        // with room for twice as many where the share allows it: the rows are copied (4.7 TB/s) a bounded number of times.  Both
        // tables are there while that is done, and the budget holds both; where it does not, room for what is needed has to do.
        size_t room = std::max(need, std::min(most, 2 * (size_t)capacity));
        if (!make_room(room * row_bytes, 0)) {
            room = need;
            if (!make_room(room * row_bytes, 0)) return false;
        }
        const size_t bytes = room * row_bytes;
        affine_t* out = nullptr;
        const int rc = grape_malloc((void**)&out, bytes);
        if (rc == GRAPE_ENOMEM) return false;
        check(rc, "grape_malloc");
        check(grape_memcpy_d2d(out, table, (size_t)rows * row_bytes, nullptr), "grape_memcpy_d2d");
        release_scaled_table(table);
        scaled_bytes_ += bytes;
        it = scaled_registry().emplace(out, ScaledTable{this, bytes, false}).first;
        table = out;
        capacity = (uint)room;
    }
    it->second.extended = true;
    const int rc = gen_scaled(reinterpret_cast<affine_t*>(reinterpret_cast<char*>(table) + (size_t)rows * row_bytes), more, ncols);
    if (rc == GRAPE_ENOMEM) return false;
    check(rc, "grape_g1_scaled_table_gen");
    return true;
}

void Hyrax::release_scaled_table(affine_t* table) {
    if (!table) return;
    auto it = scaled_registry().find(table);
    if (it != scaled_registry().end()) {
        if (it->second.owner) it->second.owner->scaled_bytes_ -= it->second.bytes;
        scaled_registry().erase(it);
    }
    grape_free(table);
}

bool Hyrax::owns_scaled_table(const affine_t* table) const {
    auto it = scaled_registry().find(table);
    return it != scaled_registry().end() && it->second.owner == this;
}

affine_t* Hyrax::commit_indexed_affine(int* idx_plus1, uint size, uint N, affine_t* scaled_table, uint ncols, uint len, int* d_flag, int base1,
                                       const void* start, bool uneven) {
    check_shape(size, N);
    const uint rowlen = N * com_scale;
    if (rowlen > ncols) throw std::runtime_error("row longer than the scaled table");
    const uint rows = size / rowlen;
    affine_t* out = nullptr;
    check(grape_malloc((void**)&out, sizeof(affine_t) * (size_t)rows), "grape_malloc");
    check(for_row_chunks(size, rowlen, [&](size_t e0, size_t n, size_t r0) {
              return grape_commit_indexed(W(out + r0), idx_plus1 + e0, n, rowlen, W(scaled_table), ncols, len, base1, static_cast<const uint32_t*>(start), uneven, d_flag, nullptr);
          }),
          "grape_commit_indexed");
    return out;
}

affine_t* Hyrax::commit_sparse_affine(FrTensor& tensor, int* skip, uint size, uint N, uint64_t live, const int* idx1) {
    check_shape(size, N);
    const uint rowlen = N * com_scale;
    const uint rows = size / rowlen;
    // From 512 live elements a row the strided table is the better one: 16 to 18 additions per element instead of 20 and four waves
    // or more on a row instead of one, against 64 partial sums per residue and row (64 GiB table; rows of 11008 padded to
    // 16384, 67 % live: 2^25 elements 53 against 93 ms, 2^21 elements 5.3 against 13.3; a quarter live, scattered: 20.6 against 26.3
    // and 1.8 against 3.8; 27 live elements a row: the queue of half waves over the per-window table).  Building it takes as long as
    // two such proofs of 2^25 elements save, and its memory: it is built once the proofs of this object would have saved as
    // much, so that a program with a few short proofs never pays for it.  Saved are 1.7 ns a live element where the
    // rows fill the chip, and 2.5 us for each live element of a row where the longest row is what takes the time.
    bool strided = false;
    if (live >= (uint64_t)512 * rows && rows > 1) {
        strided = ensure_strided_table(rowlen, false);
        if (!strided) {
            sparse_saving_ms_ += std::max(1.7e-6 * (double)live, 2.5e-3 * (double)live / rows);
            strided = ensure_strided_table(rowlen, true, &sparse_saving_ms_);
            if (strided) sparse_saving_ms_ = 0;
        }
    }
    if (strided) {
        const StridedTable& t = fr_strided_;
        affine_t* out = nullptr;
        check(grape_malloc((void**)&out, sizeof(affine_t) * (size_t)rows), "grape_malloc");
        check(for_row_chunks(size, rowlen, [&](size_t e0, size_t n, size_t r0) {
                  if (idx1)
                      return grape_commit_fr_strided_masked_indexed(W(out + r0), W(tensor.gpu_data), idx1 + e0, skip + e0, n, rowlen, W(t.d), t.ngen, t.c, t.J,
                                                                    t.nsets, nullptr);
                  return grape_commit_fr_strided_masked(W(out + r0), W(tensor.gpu_data + e0), skip + e0, n, rowlen, W(t.d), t.ngen, t.c, t.J, t.nsets, nullptr);
              }),
              "grape_commit_fr_strided_masked");
        return out;
    }
    if (!ensure_fr_table(rowlen, false)) return nullptr;
    const WideTable& t = fr_table_;
    affine_t* out = nullptr;
    check(grape_malloc((void**)&out, sizeof(affine_t) * (size_t)rows), "grape_malloc");
    check(for_row_chunks(size, rowlen, [&](size_t e0, size_t n, size_t r0) {
              if (idx1)
                  return grape_commit_fr_sparse_indexed(W(out + r0), W(tensor.gpu_data), idx1 + e0, skip + e0, n, rowlen, W(t.d), t.ngen, t.c, t.nw, t.K, nullptr);
              return grape_commit_fr_sparse(W(out + r0), W(tensor.gpu_data + e0), skip + e0, n, rowlen, W(t.d), t.ngen, t.c, t.nw, t.K, nullptr);
          }),
          "grape_commit_fr_sparse");
    return out;
}

void single_commit(fr_t* d, affine_t* g, jacob_t* com, uint N, uint npoints) {
    grape_host::ensure_init();
    affine_t* a = nullptr;
    check(grape_malloc((void**)&a, sizeof(affine_t)), "grape_malloc");
    check(grape_commit_fr_ref_table(W(a), W(d), N, N, W(g), npoints, nullptr), "grape_commit_fr_ref_table");
    check(grape_g1_affine_to_jacobian(W(com), W(a), 1, nullptr), "grape_g1_affine_to_jacobian");
    check(grape_stream_sync(nullptr), "sync");
    grape_free(a);
}

static jacob_t* to_jacobian(affine_t* aff, uint rows) {
    jacob_t* out = nullptr;
    check(grape_malloc((void**)&out, sizeof(jacob_t) * (size_t)rows), "grape_malloc");
    check(grape_g1_affine_to_jacobian(W(out), W(aff), rows, nullptr), "grape_g1_affine_to_jacobian");
    check(grape_stream_sync(nullptr), "sync");
    grape_free(aff);
    return out;
}
jacob_t* Hyrax::commit(int* tensor, uint size, uint N) {
    affine_t* a = commit_affine(tensor, size, N);
    return to_jacobian(a, size / (N * com_scale));
}
jacob_t* Hyrax::commit(FrTensor& tensor, uint size, uint N) {
    affine_t* a = commit_affine(tensor, size, N);
    return to_jacobian(a, size / (N * com_scale));
}

namespace {
// The commitment of a single row is a short accumulation and then a latency chain, so it runs on a stream of its own beside
// what the default stream works on.  The row is made or uploaded on the default stream; nothing may write to it until wait().
struct SideRow {
    static grape_stream_t stream;                 // lives as long as the process, like the event
    static void* row_there;
    struct Result { affine_t p; int flag[4]; };
    static_assert(sizeof(Result) == sizeof(affine_t) + 16, "point and flag travel together");
    Result* d = nullptr;
    bool open = false;
    SideRow() {
        if (!stream) {
            check(grape_stream_create(&stream), "grape_stream_create");
            check(grape_stream_internal(stream), "grape_stream_internal");
            check(grape_event_create(&row_there), "grape_event_create");
        }
        check(grape_event_record(row_there, nullptr), "grape_event_record");        // a short row travels as a queued launch
        check(grape_stream_wait_event(stream, row_there), "grape_stream_wait_event");
        check(grape_malloc((void**)&d, sizeof(Result)), "grape_malloc");
        open = true;
        check(grape_memset_zero(d->flag, sizeof(int), stream), "grape_memset_zero");
    }
    ~SideRow() {
        if (open) grape_stream_sync(stream);      // left by an exception: nothing the stream still reads is freed under it
        grape_free(d);
    }
    affine_t wait(bool flag_used) {
        Result h;
        check(grape_memcpy_d2h(&h, d, sizeof h, stream), "d2h");
        open = false;
        if (flag_used && h.flag[0]) throw std::runtime_error("Hyrax: a scalar of a single row does not fit the table's digit range");
        return h.p;
    }
};
grape_stream_t SideRow::stream = nullptr;
void* SideRow::row_there = nullptr;
}  // namespace

// Hyrax::open, src/Hyrax.cu:237-305: fold the tensor down to one row x of length new_N at the
// outer variables of the point, blind it as z = c*x + d with a random row d, commit d, and send
// <a,d>*G where a is the eq-vector of the inner variables.
Hyrax_proof Hyrax::open(FrTensor& tensor, const std::vector<Fr> eval_point_, Fr c, uint size, uint N) {
    return open_impl(&tensor, nullptr, eval_point_, c, size, N);
}
Hyrax_proof Hyrax::open(const int* device_int_data, const std::vector<Fr> eval_point_, Fr c, uint size, uint N) {
    return open_impl(nullptr, device_int_data, eval_point_, c, size, N);
}
// tensor_in, or the integer tensor `ints` read as FrTensor::get_data would embed it: its fold over the rows then reads the
// integers directly (4 bytes per element where embedding and folding move 68)
Hyrax_proof Hyrax::open_impl(FrTensor* tensor_in, const int* ints, const std::vector<Fr>& eval_point_, Fr c, uint size, uint N) {
    if (size / N / com_scale < layer_num) throw std::runtime_error("Size too small: size < N * com_scale * layer_num");
    uint pad_N = 1u << Log2(N);
    uint new_N = pad_N * com_scale;
    assert(eval_point_.size() == Log2(size));
    last_open_point_ = eval_point_;
    fr_t* eval_point = grape_host::upload(eval_point_, OnDefaultStream());

    FrTensor d = FrTensor::random(new_N, OnDefaultStream());

    // commitment of d (single_commit, src/Hyrax.cu:176-185) beside the folds of the tensor below, which do not write to d
    SideRow com_d;
    const bool flag_used = commit_fr_rows(&com_d.d->p, d.gpu_data, new_N, new_N, false, SideRow::stream, com_d.d->flag);

    std::unique_ptr<FrTensor> rows_of_ints;
    if (ints) {
        rows_of_ints.reset(new FrTensor(FrTensor::folded_from_ints(ints, size, eval_point, (size / layer_num) / (N * com_scale),
                                                                    Log2(N * com_scale), N * com_scale, OnDefaultStream())));
    } else {
        tensor_in->partial_eval(size, eval_point, (size / layer_num) / (N * com_scale), Log2(N * com_scale), N * com_scale);
    }
    FrTensor& tensor = ints ? *rows_of_ints : *tensor_in;
    tensor.partial_eval((N * com_scale) * layer_num, eval_point, layer_num, Log2(size / layer_num), N * com_scale);
    // x, the row that is left (padded): a copy where the tensor is the caller's, which is bound to its last element
    std::unique_ptr<FrTensor> row;
    if (!ints || pad_N != N) {
        row.reset(new FrTensor(new_N, OnDefaultStream()));
        if (pad_N == N) {
            *row = tensor;
        } else {
            // padded from where it lies: neither the folded integers nor a single row hold the padded length, which pad() would write there
            check(grape_fr_pad(W(row->gpu_data), W(tensor.gpu_data), N, pad_N, new_N, W(grape_host::device_scalar(Fr::zero())), nullptr), "grape_fr_pad");
        }
    }
    const FrTensor& x = row ? *row : tensor;

    // z = c x + d, and behind it <a, x> and <a, d>: two evaluations at the inner variables side by side, read with z by one copy
    const size_t behind = grape_fr_fold_i32_elems(new_N, new_N, 1);
    FrTensor z((uint)(new_N + 2 * behind), OnDefaultStream());
    const fr_t* const at_x = z.gpu_data + new_N;
    grape_fold_job folds[2] = {};
    for (uint k = 0; k < 2; k++) {
        folds[k].t = W(z.gpu_data + new_N + k * behind);
        folds[k].from = W(k ? d.gpu_data : x.gpu_data);
        folds[k].N = folds[k].c = new_N;
        folds[k].x = W(eval_point);
        folds[k].gap = 1;
    }
    check(grape_fr_fold_pair(folds, 2, nullptr), "grape_fr_fold_pair");
    check(grape_fr_axpy(W(z.gpu_data), W(d.gpu_data), W(grape_host::device_scalar(c)), W(x.gpu_data), new_N, nullptr), "grape_fr_axpy");
    if (!ints) check(grape_memcpy_d2d(tensor.gpu_data, at_x, sizeof(fr_t), nullptr), "grape_memcpy_d2d");
    std::vector<Fr> zs(new_N + behind + 1);
    check(grape_memcpy_d2h(zs.data(), z.gpu_data, sizeof(fr_t) * zs.size(), nullptr), "d2h");
    const Fr result = zs[new_N];
    bn128 commit_ad = multiple_of_G(zs[new_N + behind]);

    const affine_t host_com_d = com_d.wait(flag_used);
    grape_free_on_default(eval_point);
    Hyrax_proof proof(result, new_N, bn128(host_com_d), commit_ad);
    std::copy(zs.begin(), zs.begin() + new_N, proof.z);
    return proof;
}

// The driver-side verification of test/HyraxTest.cu:87-125: fold the row commitments at the outer
// variables, then check  c*C + com_d == com(z)  and  (c*result)*G + com_ad == <a,z>*G.
bool Hyrax::verify(Hyrax_proof& proof, jacob_t* commitment, const std::vector<Fr>& eval_point, Fr c, uint size, uint N) {
    const uint rowlen = N * com_scale;
    const uint rows = size / rowlen;
    const uint new_N = (uint)proof.z_size;
    const uint inner = Log2(rowlen);
    // com(z) beside everything else
    std::vector<Fr> zv(proof.z, proof.z + new_N);
    FrTensor z = FrTensor::from_host(zv, OnDefaultStream());
    SideRow com_z_row;
    const bool flag_used = commit_fr_rows(&com_z_row.d->p, z.gpu_data, new_N, new_N, false, SideRow::stream, com_z_row.d->flag);
    // c * C, C the row commitments folded at the outer variables: sum_i c eq(outer, i) C_i, its window sums on the device
    // and their doubling chain here.  (Folding fewer variables than the rows need leaves the first 2^variables rows; each
    // variable beyond them finds the rows above missing, a factor 1 - u, and needs no table.)
    std::vector<Fr> outer(eval_point.begin() + inner, eval_point.end());
    Fr scale = c;
    for (; outer.size() > Log2(rows); outer.pop_back()) scale *= Fr::one() - outer.back();
    const uint used = ((uint64_t)1 << outer.size()) < rows ? 1u << outer.size() : rows;
    FrTensor pyramid((uint)grape_eq_pyramid_elems((uint)outer.size()), OnDefaultStream());
    fr_t* d_outer = grape_host::upload(outer, OnDefaultStream());
    check(grape_eq_pyramid(W(pyramid.gpu_data), W(d_outer), (uint)outer.size(), nullptr), "grape_eq_pyramid");
    grape_free_on_default(d_outer);
    fr_t* const weights = pyramid.gpu_data + (((size_t)1 << outer.size()) - 1);
    check(grape_fr_bcast_mul(W(weights), W(weights), W(grape_host::device_scalar(scale)), (size_t)1 << outer.size(), nullptr), "grape_fr_bcast_mul");
    // the window sums and behind them <a, z>, read by one copy
    struct { bucket_t windows[GRAPE_MSM_WINDOWS]; Fr az; } got;
    static_assert(sizeof(got) == sizeof(bucket_t) * GRAPE_MSM_WINDOWS + sizeof(Fr), "read as it lies there");
    std::vector<Fr> inner_point(eval_point.begin(), eval_point.begin() + inner);
    const bool plain = ((uint64_t)1 << inner) == new_N;
    const size_t behind = plain ? grape_fr_fold_i32_elems(new_N, new_N, 1) : 0;
    char* d_got = nullptr;
    check(grape_malloc_on_default((void**)&d_got, sizeof(got.windows) + sizeof(Fr) * (behind + 1)), "grape_malloc");
    check(grape_g1_msm_windows(W(d_got), W(commitment), W(weights), used, nullptr), "grape_g1_msm_windows");
    if (plain) {
        fr_t* d_inner = grape_host::upload(inner_point, OnDefaultStream());
        check(grape_fr_fold_from(W(d_got + sizeof(got.windows)), W(z.gpu_data), new_N, W(d_inner), new_N, 0, 1, nullptr), "grape_fr_fold_from");
        grape_free_on_default(d_inner);
    }
    check(grape_memcpy_d2h(&got, d_got, plain ? sizeof(got) : sizeof(got.windows), nullptr), "grape_memcpy_d2h");
    grape_free_on_default(d_got);
    bucket_t cC = got.windows[GRAPE_MSM_WINDOWS - 1];
    for (int w = GRAPE_MSM_WINDOWS - 2; w >= 0; w--) {
        for (int d = 0; d < 4; d++) grape::xyzz_dbl(cC);
        grape::xyzz_add(cC, got.windows[w]);
    }
    const affine_t com_z = com_z_row.wait(flag_used);
    if (!(bn128(grape::xyzz_to_jac(cC)) + proof.commit_d == bn128(com_z))) return false;
    // (c * result) * G + commit_ad == az * G, with one multiple of G
    const Fr az = plain ? got.az : z(inner_point);
    return proof.commit_ad == multiple_of_G(az - c * proof.result);
}

// G is a member that a caller may set: the multiples are made anew for another one
bn128 Hyrax::multiple_of_G(const Fr& k) {
    if (!G_multiples_ || std::memcmp(&G_multiples_of_, &G, sizeof G) != 0) {
        G_multiples_.reset(new G1FixedBase(G));
        G_multiples_of_ = G;
    }
    return G_multiples_->mul(k);
}

void Hyrax::verify(Hyrax_proof& proof, jacob_t* commitment, Fr c, uint size, uint N) {
    if (last_open_point_.size() != Log2(size)) throw std::runtime_error("Hyrax::verify: no opening of this size was made by this object");
    if (!verify(proof, commitment, last_open_point_, c, size, N)) throw std::runtime_error("Hyrax::verify: the opening does not match the commitment");
}
