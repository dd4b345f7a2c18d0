// Launch geometry and address arithmetic of the wide-table commitment kernels, in one place so that
// the kernels, their launcher and a host build (tests/native/commit_geometry_host.cpp, which walks
// every wave of a shape and checks each offset against the size of the buffer it indexes) run the
// same expressions.  All element counts and offsets are size_t; only per-row quantities are 32-bit.
#pragma once
#include <stddef.h>
#include <stdint.h>
#include "field.hpp"

namespace grape {
namespace geom {

constexpr int kPartialWords = 64;      // one lane's partial accumulator: 256 bytes
constexpr int kWaveLanes = 64;
constexpr size_t kSlabSegments = 32768;   // row segments per launch: 512 MiB of partial sums

// Bounds the column segments of a row (wide_plan): a row leaves at most 128 partial sums per 2^this.
GRAPE_HD uint32_t reduce_lanes_log2(size_t rows) {
    if (rows >= 2048) return 3;
    if (rows >= 1024) return 4;
    if (rows >= 512) return 5;
    return 6;
}

struct WidePlan {
    size_t rows;            // size / rowlen
    uint32_t lg_lpr;        // reduce_lanes_log2 of the rows
    uint32_t nseg, seg;     // column segments per row and their length
    size_t slab;            // rows per launch
    size_t partial_bytes;   // work buffer of one launch (slab * nseg * 64 lanes * 256 bytes)
};
// segments: two waves per SIMD (one with fewer than 512 rows: there the additions of the row reduction cost as much as
// those saved by shorter lane chains - 64 rows of 4096: 159 us in 16 segments, 184 in 32, 252 in 64; 256 rows 284, 292,
// 339; 512 rows 447, 439, 478; 1024 rows 764, 720, 723), at least 64 columns per lane-sweep, and no more than
// leaves 128 * 2^lg_lpr partial sums per row; rows go through in slabs of slab_segments row segments
GRAPE_HD WidePlan wide_plan(size_t size, uint32_t rowlen, size_t slab_segments) {
    WidePlan p;
    p.rows = size / rowlen;
    p.lg_lpr = reduce_lanes_log2(p.rows);
    p.nseg = 1;
    const size_t waves = p.rows < 512 ? 1024 : 2048;
    while (p.rows * p.nseg < waves && rowlen / (p.nseg * 2) >= 64 && p.nseg * 2 <= (2u << p.lg_lpr)) p.nseg *= 2;
    p.seg = (rowlen + p.nseg - 1) / p.nseg;
    p.slab = slab_segments / (size_t)p.nseg;
    if (p.slab < 1) p.slab = 1;
    if (p.slab > p.rows) p.slab = p.rows;
    p.partial_bytes = p.slab * p.nseg * kWaveLanes * (size_t)(4 * kPartialWords);
    return p;
}

// Windows of full-width scalars over several waves: a call with few rows runs one wave per SIMD or less, each lane a chain of
// one addition (10 us) per window.  Up to 1024 waves take shares of the windows, the partial sums they leave more
// cost the row reduction a level of groups (one row of 4096 with 20 windows: 354 -> 232 us; 16 rows
// 386 -> 377; one row of 256 with 15 windows 289 -> 139, 64 rows 301 -> 163).  With 1024 waves and more the chip is busy and nothing is split.
struct WindowSplit {
    uint32_t parts, per;    // shares per (row, segment) and windows in each
};
GRAPE_HD WindowSplit window_split(size_t waves, uint32_t nwin) {
    const size_t room = waves ? 1024 / waves : 1;
    WindowSplit w;
    w.parts = room < 1 ? 1 : room < nwin ? (uint32_t)room : nwin;
    w.per = (nwin + w.parts - 1) / w.parts;
    w.parts = (nwin + w.per - 1) / w.per;
    return w;
}

// what wave `wave` of a launch over `rows` rows works on
struct WaveSpan {
    size_t row;
    uint32_t s, col_end;
};
GRAPE_HD WaveSpan wave_span(size_t wave, uint32_t nseg, uint32_t seg, uint32_t rowlen) {
    WaveSpan w;
    w.row = wave / nseg;
    w.s = (uint32_t)(wave - w.row * nseg);
    w.col_end = (w.s + 1) * seg < rowlen ? (w.s + 1) * seg : rowlen;
    return w;
}
// element index of scalar (row, col) of a launch whose scalar pointer starts at its first row
GRAPE_HD size_t scalar_index(size_t row, uint32_t rowlen, uint32_t col) { return row * rowlen + col; }
// entry index of digit magnitude mag (1..K) of window w for generator col in a table over N generators
GRAPE_HD size_t table_entry(uint32_t w, uint32_t K, uint32_t mag, size_t N, uint32_t col) {
    return ((size_t)w * K + (mag - 1)) * N + col;
}
// 32-bit-word offset of partial accumulator i (i = wave * 64 + lane in the accumulation kernel,
// row * nparts + j in the reduction kernel)
GRAPE_HD size_t partial_word(size_t i) { return (size_t)kPartialWords * i; }
// row of lane `lane` of wave `wave` when 2^lg_lpr lanes share a row
GRAPE_HD size_t reduce_row(size_t wave, int lane, uint32_t lg_lpr) { return wave * (size_t)(kWaveLanes >> lg_lpr) + (size_t)(lane >> lg_lpr); }
// which share of its row the quad of lane `lane` takes
GRAPE_HD uint32_t quad_share(int lane, uint32_t lg_qpr) { return (uint32_t)(lane >> 2) & ((1u << lg_qpr) - 1u); }

// How a row's nparts partial sums become one (measured with the three kernels of g1_kernels.hip, microseconds):
//   - more than 8192 rows: lanes first, down to 8 per row, then quads (32768 rows of 64: 540, quads alone 650 to 680);
//     at 8192 rows quads alone are as fast (209 against 199) and one launch less;
//   - up to 512 rows of more than 64 partial sums: quads in groups of 64 first, so that the chain stays at 7 additions
//     (512 rows of 512: 196 against 243; 64 of 4096: 223 against 1430; 1024 rows of 256: 190 against 162, so not there);
//     and again in groups of 16 where that leaves more than 64 (rows whose windows were split);
//   - quads per row: as many as a wave holds while rows * quads stays below 2^15, i.e. two waves per SIMD (2048 rows
//     of 128: 154 with 16, 151 with 8, 232 with 4; 8192 of 64: 285, 225, 209 with 16, 8, 4).
constexpr uint32_t kQuadsPerWaveLog2 = 4;
constexpr uint32_t kReduceGroup = 64;      // partial sums of a group
constexpr uint32_t kReduceGroup2 = 16;     // and of a group of groups
constexpr uint32_t kReduceKeep = 8;        // partial sums per row that the lane kernel leaves
struct ReducePlan {
    bool lanes;             // first stage by commit_reduce_lane_kernel
    uint32_t left;          // partial sums per row after the first stage (nparts when there is none)
    uint32_t left2;         // and after the second (left when there is none)
    uint32_t lg_qpr;        // log2 of the quads per row in the last stage
};
GRAPE_HD ReducePlan reduce_plan(size_t rows, uint32_t nparts) {
    ReducePlan p;
    p.lanes = rows > 8192 && nparts > kReduceKeep;
    p.left = p.lanes ? kReduceKeep : (rows <= 512 && nparts > kReduceGroup && nparts % kReduceGroup == 0) ? nparts / kReduceGroup : nparts;
    p.left2 = !p.lanes && p.left < nparts && p.left > kReduceGroup && p.left % kReduceGroup2 == 0 ? p.left / kReduceGroup2 : p.left;
    p.lg_qpr = 0;
    while (p.lg_qpr < kQuadsPerWaveLog2 && (2u << p.lg_qpr) <= p.left2 && (rows << (p.lg_qpr + 1)) <= 32768) p.lg_qpr++;
    if (p.lanes) p.lg_qpr = 1;
    return p;
}
// accumulators of work space for at most `rows` rows: what the first two stages leave, and the row sums
GRAPE_HD size_t reduce_tmp_accumulators(size_t rows, uint32_t nparts) {
    const size_t groups = nparts / kReduceGroup, grouped = (rows < 512 ? rows : 512) * (groups + groups / kReduceGroup2), kept = rows > 8192 ? rows * kReduceKeep : 0;
    return rows + (grouped > kept ? grouped : kept);
}

// The launches of a reduction, in order.  A stage reads `units` times `parts` accumulators (the partial sums for the first stage,
// work space from accumulator `from` on otherwise) and leaves one per unit (`keep` per unit for the lane kernel) in work
// space from accumulator `to` on; the last stage's are the row sums.
struct ReduceStage {
    bool lanes;             // commit_reduce_lane_kernel, else commit_reduce_quad_kernel
    size_t units;
    uint32_t parts, keep, lg_qpr;
    size_t from, to;
};
constexpr int kMaxReduceStages = 3;
GRAPE_HD int reduce_stages(size_t rows, uint32_t nparts, ReduceStage* st) {
    const ReducePlan p = reduce_plan(rows, nparts);
    int n = 0;
    size_t from = 0, used = 0;
    if (p.lanes) st[n++] = ReduceStage{true, rows, nparts, p.left, 0, 0, 0};
    else if (p.left < nparts) st[n++] = ReduceStage{false, rows * p.left, nparts / p.left, 1, kQuadsPerWaveLog2, 0, 0};
    if (n) used = rows * p.left;
    if (p.left2 < p.left) {
        st[n++] = ReduceStage{false, rows * p.left2, p.left / p.left2, 1, kQuadsPerWaveLog2, from, used};
        from = used;
        used += rows * p.left2;
    }
    st[n++] = ReduceStage{false, rows, p.left2, 1, p.lg_qpr, from, used};
    return n;
}
// row and first partial sum of thread `t` of the lane kernel (it goes on in steps of `keep`)
GRAPE_HD size_t lane_row(size_t t, uint32_t keep) { return t / keep; }
GRAPE_HD uint32_t lane_share(size_t t, uint32_t keep) { return (uint32_t)(t % keep); }

// Workgroups are dealt to the chip's 32 shader engines in turn (workgroup i to XCD i mod 8, and in turn within it), whether
// or not that engine has room.  Where the work of a unit depends on its position - rows of 11008 padded to 16384 leave
// every fourth committed row empty - units in launch order leave whole engines idle.  spread_unit is a permutation
// of 0 .. n - 1 under which every engine's workgroups sweep all positions: engine a = i mod 32 takes the a-th stretch of
// n / 32 steps of a walk with stride `step`, a number near the golden section of n and prime to it.
// (2^25 full-width scalars on such rows: 73.4 ms in launch order, 56.6 this way, 79 to 81 with no row empty.)
GRAPE_HD size_t spread_unit(size_t i, size_t n, size_t step) {
    const size_t whole = n >> 5;
    if (i >= whole << 5) return i;
    return (((i & 31) * whole + (i >> 5)) * step) % (whole << 5);
}
inline size_t spread_step(size_t n) {
    const size_t m = n >> 5 << 5;
    size_t step = (size_t)(0.6180339887 * (double)m) | 1;
    for (;; step += 2) {
        size_t a = m, b = step;
        while (b) {
            const size_t r = a % b;
            a = b;
            b = r;
        }
        if (a == 1 || m == 0) return step;
    }
}
// workgroups of a launch of `threads` threads in groups of `per_block`
GRAPE_HD size_t blocks_needed(size_t threads, size_t per_block) { return (threads + per_block - 1) / per_block; }

}  // namespace geom
}  // namespace grape
