// Host walk over the launch geometry of the wide-table commitment (grape_amd/csrc/commit_geometry.hpp,
// the expressions the kernels and their launcher use): every wave of every launch of a shape, its
// scalar reads, table gathers, the windows it takes, its partial-sum stores, every stage of the row
// reduction with its loads and stores in the partial sums and the work space, and the output rows,
// each offset checked against the size of the buffer it indexes, every partial sum counted (each is
// added once), every grid against the 32-bit limits of a launch.  Returns the number of violations; report[] receives the first one.
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <vector>
#include "../../grape_amd/csrc/commit_geometry.hpp"
using namespace grape;

namespace {
struct Checker {
    long long bad = 0;
    char* report;
    size_t cap;
    void fail(const char* what, size_t got, size_t limit) {
        if (bad == 0 && report) snprintf(report, cap, "%s: %zu >= %zu", what, got, limit);
        bad++;
    }
    void lt(const char* what, size_t got, size_t limit) { if (!(got < limit)) fail(what, got, limit); }
    void le(const char* what, size_t got, size_t limit) { if (!(got <= limit)) fail(what, got, limit + 1); }
};
// The stages that launch_reduce queues for `rows` rows of `nparts` partial sums each, in work space sized for slabs of `slab` rows.
void reduce_walk(Checker& ck, size_t slab, size_t rows, uint32_t nparts, size_t partial_words) {
    geom::ReduceStage st[geom::kMaxReduceStages];
    const int n = geom::reduce_stages(rows, nparts, st);
    const size_t tmp = geom::reduce_tmp_accumulators(slab, nparts);
    ck.le("stages of a reduction", (size_t)n, geom::kMaxReduceStages);
    size_t held = rows * nparts;                                        // accumulators that the stage before left
    for (int i = 0; i < n; i++) {
        const geom::ReduceStage& g = st[i];
        if (g.units * g.parts != held) ck.fail("accumulators taken by a stage", g.units * g.parts, held);
        if (i && g.from != st[i - 1].to) ck.fail("source of a stage", g.from, st[i - 1].to);
        // a stage must not write where it reads
        if (i && g.to < g.from + held && g.from < g.to + g.units * g.keep) ck.fail("a stage writes what it reads", g.to, g.from + held);
        std::vector<unsigned char> taken(held, 0);
        size_t stored = 0;
        auto load = [&](size_t row, uint32_t j) {
            const size_t at = row * g.parts + j;
            ck.lt("accumulator loaded", at, held);
            if (at < held) taken[at]++;
            if (i == 0) ck.lt("partial word (load)", geom::partial_word(at) + geom::kPartialWords - 1, partial_words);
            else ck.lt("work space (load)", g.from + at, tmp);
        };
        auto store = [&](size_t at) {
            ck.lt("accumulator stored", at, g.units * g.keep);
            ck.lt("work space (store)", g.to + at, tmp);
            stored++;
        };
        const size_t threads = g.lanes ? g.units * g.keep : g.units << (g.lg_qpr + 2);
        const size_t blocks = geom::blocks_needed(threads, 256);
        ck.le("reduction grid (workgroups)", blocks, 0x7fffffffull);
        ck.le("reduction grid (threads)", blocks * 256, 0xffffffffull);
        if (g.lanes) {
            for (size_t t = 0; t < blocks * 256; t++) {
                if (t >= g.units * g.keep) continue;                    // the kernel's own exit
                for (uint32_t j = geom::lane_share(t, g.keep); j < g.parts; j += g.keep) load(geom::lane_row(t, g.keep), j);
                store(t);
            }
        } else {
            ck.le("quads of a row", (size_t)4 << g.lg_qpr, geom::kWaveLanes);
            for (size_t wave = 0; wave < blocks * 4; wave++) {
                for (int lane = 0; lane < geom::kWaveLanes; lane += 4) {
                    const size_t row = geom::reduce_row(wave, lane, g.lg_qpr + 2);
                    const uint32_t sub = geom::quad_share(lane, g.lg_qpr);
                    for (int l = 1; l < 4; l++)
                        if (geom::reduce_row(wave, lane + l, g.lg_qpr + 2) != row || geom::quad_share(lane + l, g.lg_qpr) != sub)
                            ck.fail("the lanes of a quad", lane + l, lane);
                    if (row >= g.units) continue;
                    for (uint32_t j = sub; j < g.parts; j += 1u << g.lg_qpr) load(row, j);
                    if (sub == 0) store(row);
                }
            }
        }
        for (size_t k = 0; k < held; k++)
            if (taken[k] != 1) ck.fail("times an accumulator is added", taken[k], 1);
        if (stored != g.units * g.keep) ck.fail("accumulators stored", stored, g.units * g.keep);
        held = g.units * g.keep;
    }
    if (held != rows) ck.fail("row sums", held, rows);
}
// every window of a scalar in exactly one share
void window_walk(Checker& ck, const geom::WindowSplit& split, uint32_t nwin) {
    std::vector<unsigned char> taken(nwin, 0);
    for (uint32_t part = 0; part < split.parts; part++) {
        ck.lt("first window of a share", part * split.per, nwin);
        for (uint32_t w = part * split.per; w < (part + 1) * split.per && w < nwin; w++) taken[w]++;
    }
    for (uint32_t w = 0; w < nwin; w++)
        if (taken[w] != 1) ck.fail("times a window is taken", taken[w], 1);
}
}  // namespace

extern "C" long long reduce_geometry_check(size_t slab, size_t rows, uint32_t nparts, char* report, size_t report_cap) {
    Checker ck{0, report, report_cap};
    if (report && report_cap) report[0] = 0;
    reduce_walk(ck, slab, rows, nparts, rows * nparts * (size_t)geom::kPartialWords);
    return ck.bad;
}
extern "C" long long window_split_check(size_t waves, uint32_t nwin, uint32_t* parts_out, char* report, size_t report_cap) {
    Checker ck{0, report, report_cap};
    if (report && report_cap) report[0] = 0;
    const geom::WindowSplit split = geom::window_split(waves, nwin);
    window_walk(ck, split, nwin);
    *parts_out = split.parts;
    return ck.bad;
}
// geom::spread_unit over 0 .. n - 1; units[i] receives the unit of workgroup i
extern "C" void spread_units(size_t n, size_t* units) {
    const size_t step = geom::spread_step(n);
    for (size_t i = 0; i < n; i++) units[i] = geom::spread_unit(i, n, step);
}

extern "C" long long commit_geometry_check(size_t size, uint32_t rowlen, size_t N, uint32_t nw, uint32_t K, uint32_t elem_words,
                                           size_t slab_segments, uint32_t entry_words, uint32_t point_words, size_t* partial_bytes_out,
                                           size_t* launches_out, char* report, size_t report_cap) {
    Checker ck{0, report, report_cap};
    if (report && report_cap) report[0] = 0;
    const geom::WidePlan plan = geom::wide_plan(size, rowlen, slab_segments);
    // full-width scalars of few rows: their windows over several waves
    geom::WindowSplit split = {1, nw};
    if (elem_words == 8) split = geom::window_split(plan.rows * plan.nseg, nw);
    window_walk(ck, split, nw);
    const size_t partial_bytes = plan.partial_bytes * split.parts;
    if (partial_bytes_out) *partial_bytes_out = partial_bytes;
    const size_t scalar_words = size * elem_words;                     // 32-bit words in the scalar buffer
    const size_t table_words = (size_t)nw * K * N * entry_words;
    const size_t partial_words = partial_bytes / 4;
    const size_t out_words = plan.rows * point_words;
    size_t launches = 0;
    for (size_t r0 = 0; r0 < plan.rows; r0 += plan.slab) {
        launches++;
        const size_t nr = plan.rows - r0 < plan.slab ? plan.rows - r0 : plan.slab;
        const size_t sc_base = r0 * rowlen * elem_words;               // word offset of this launch's scalars
        const size_t threads = nr * plan.nseg * split.parts * geom::kWaveLanes;
        const size_t blocks = geom::blocks_needed(threads, 256);
        ck.le("accumulation grid (workgroups)", blocks, 0x7fffffffull);
        ck.le("accumulation grid (threads)", blocks * 256, 0xffffffffull);
        const size_t waves = blocks * 4;
        for (size_t wave = 0; wave < waves; wave++) {
            if (wave >= nr * plan.nseg * split.parts) continue;         // the kernel's own exit
            const geom::WaveSpan sp = geom::wave_span(wave / split.parts, plan.nseg, plan.seg, rowlen);
            ck.lt("row of a wave", sp.row, nr);
            // first and last lane, first and last column each of them reads (incl. the two scalars kept in flight)
            for (int lane = 0; lane < geom::kWaveLanes; lane += geom::kWaveLanes - 1) {
                const uint32_t c0 = sp.s * plan.seg + (uint32_t)lane;
                if (c0 < sp.col_end) {
                    uint32_t last = c0 + ((sp.col_end - 1 - c0) / 64) * 64;
                    for (uint32_t col : {c0, last}) {
                        const size_t si = geom::scalar_index(sp.row, rowlen, col);
                        ck.lt("scalar word", sc_base + (si + 1) * elem_words - 1, scalar_words);
                        // extreme table entries this column can gather: window 0 / nw-1, magnitude 1 / K
                        ck.lt("table word", (geom::table_entry(nw - 1, K, K, N, col) + 1) * entry_words - 1, table_words);
                        ck.lt("table word (touch of the next column)", (geom::table_entry(0, K, K, N, col) + 1) * entry_words - 1, table_words);
                    }
                }
                ck.lt("partial word (store)", geom::partial_word(wave * 64 + lane) + geom::kPartialWords - 1, partial_words);
            }
        }
        reduce_walk(ck, plan.slab, nr, plan.nseg * split.parts * geom::kWaveLanes, partial_words);
        ck.le("output word", (r0 + nr) * point_words, out_words);
    }
    if (launches_out) *launches_out = launches;
    return ck.bad;
}
