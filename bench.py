#!/usr/bin/env python3
"""Benchmark of the headline metric: Hyrax row commitment of a quantised weight matrix
(benchmark configuration configs[1]) on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W]

A step is one full commitment of a 4096 x 4096 int16-range matrix (sigma = 2^10, clipped) against
4096 seeded generators through the C ABI (small-scalar fast path), inputs already resident in HBM.
The K timed steps run one after the other, each call (grape_commit_i32) waiting for its result.
The same K steps are then measured as a stream of independent commitments, queued without waiting
(grape_commit_i32_nowait) on three streams in turn so that one commitment's row reduction runs
under the next one's accumulation, and reported under "pipelined".  One JSON line is printed with the throughput in Mpoints/s (points = matrix elements),
the roofline of the dominant kernel (accumulation kernel; its duration is measured live with HIP
events on the launch stream) and the CPU oracle timed on a bounded sample of rows of the same
workload on this machine's host cores.
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.join(ROOT, "tests"))

ROWS = 4096
COLS = 4096
SIGMA = 1024.0
SEED_W = 20240001
SEED_G = 20240002
RADIX_BITS = 16        # one signed 16-bit digit per scalar
K_DIGIT = 32768

# The curve is BLS12-381 (what the benchmark configurations name) unless GRAPE_CURVE=bn254 selects
# the BN254 build of the libraries and of the oracle.
CURVE = os.environ.get("GRAPE_CURVE", "bls12_381")
FP_WORDS, FP_LIMBS30 = (8, 9) if CURVE == "bn254" else (12, 13)
# Algorithmic work per committed point, the reference's algorithm (two non-zero byte windows of an
# int16 scalar, each a mixed XYZZ addition of 8M+2S, 2n^2+n 32x32 multiplies per n-limb Montgomery
# product: 300 for the 12 limbs of BLS12-381, 136 for the 8 of BN254): 2 * 10 * 300 = 6000.
ALG_MULS_PER_POINT = 2 * 10 * (2 * FP_WORDS * FP_WORDS + FP_WORDS)
# What the fast path executes: ONE mixed addition per point on L limbs of 30 bits (L = 13 resp.
# 9): 6 products of L*L + L*L + 1 multiply-adds, one fused difference of two products
# (2*L*L + L*L + 1), 2 squares of L(L+1)/2 + L*L + 1 and 4 subtractions inside products of L - 1: 3112 for L = 13, 1508 for L = 9.
_L = FP_LIMBS30
EXEC_MULS_PER_POINT = 6 * (2 * _L * _L + 1) + (3 * _L * _L + 1) + 2 * (_L * (_L + 1) // 2 + _L * _L + 1) + 4 * (_L - 1)
# lane-level 32x32 multiplies per second if every SIMD issued one v_mad_u64_u32 per cycle:
# 256 CUs x 4 SIMDs x 16 lanes x 2.4 GHz
PEAK_MULS_NOMINAL = 256 * 64 * 2.4e9
HBM_PEAK_GBPS = 8000.0
# HBM bytes per launch read from hardware counters (FETCH_SIZE + WRITE_SIZE, each scaled by what the
# same counter reads for the 1 GiB copy kernel below); the counters cannot be read from inside this
# process, so these are the figures of the committed counter summary of this same command.
COMMIT_KERNEL_TRAFFIC_BYTES = 2.627e9
FOLD_KERNEL_TRAFFIC_BYTES = 1.110e9


def gaussian_i16(shape, seed, sigma=SIGMA):
    rng = np.random.default_rng(seed)
    x = np.rint(rng.normal(0.0, sigma, size=shape))
    return np.clip(x, -32768, 32767).astype(np.int32)


def seeded_scalars(n, seed):
    """n canonical scalars < r from a seeded generator (rejection sampling of 255-bit draws)."""
    from gpuutil import rand_fr
    return rand_fr(n, seed)


def cpu_baseline(W, gens_dev, ops, budget_s=15.0):
    """The CPU oracle (reference algorithm: byte-window table, OpenMP over rows) on a bounded
    sample of rows of the same matrix; also checks the GPU result of those rows."""
    import orc
    table_dev = ops.g1_table_gen(gens_dev, 256)
    ops.sync()
    table = ops.g1_to_host(table_dev)          # 256 x 4096 affine points, the reference's table format
    del table_dev
    threads = orc.lib().orc_num_threads()
    probe = max(threads, 8)
    t0 = time.perf_counter()
    first = orc.commit_i32(W[:probe], table, COLS, COLS)
    dt = time.perf_counter() - t0
    rows = int(min(ROWS, max(probe, (budget_s / max(dt, 1e-6)) * probe)))
    rows -= rows % probe
    rows = max(rows, probe)
    t0 = time.perf_counter()
    out = orc.commit_i32(W[:rows], table, COLS, COLS)
    dt = time.perf_counter() - t0
    assert np.array_equal(out[:probe], first)
    return {"value": rows * COLS / dt / 1e6, "unit": "Mpoints/s", "cores": threads, "kind": "port",
            "sample": "first %d of %d rows (x %d columns) of the same matrix, %.1f s" % (rows, ROWS, COLS, dt)}, out


def layer_workload(args):
    """Benchmark configuration configs[4]: one LLaMA-2-7B-shape decoder layer (d_model 4096, 32 heads of 128,
    FFN 11008, seq_len 2048 by default) proved on one GPU with seeded synthetic int16 weights and
    fresh activations per layer: Hyrax commitments of the 7 weight matrices, matmul sumchecks for
    Q/K/V/O/gate/up/down and per-head QK^T / AV, range lookups on every rescaling remainder, mapping
    lookups for the softmax exponential and SiLU, and the openings the reference's driver runs beside
    them.  Witnesses (exact integer products, quotients, remainders) come from the library's integer
    kernels (--witness native, default) or from torch (--witness torch), as the reference produces its
    own with a Python model; all proving goes through the C++ host classes.

    The figure is taken like the reference's total_prove_time (test/llm.cu:69-125): the wall clock of
    every proof block between two device synchronisations, a block running from the integer tensors
    (their embedding into Fr, the deep copies, the evaluation of the quotient that forms the claim)
    through the sub-proof to the Hyrax opening that the driver checks it against.  A product
    Y = A.B^T = q*2^16 + r is proved as there: range lookup on r at the product's point u with the
    opening of r (the two must agree), claim = q(u)*2^16 + r(u), matmul sumcheck on that claim, opening
    of the weight at the reassembled point (must equal the sumcheck's final value of B).  The sum of
    the provers' own timers (what this figure was before) is kept as provers_only_s.
    One step = one whole layer; prints one JSON line."""
    import torch
    from grape_amd import ops, _host as host
    from gpuutil import rand_fr
    ops.init(0)
    host.load()
    host.load().grape_host_seed(12345)          # seeds the host classes' challenge generator
    host.set_input_format("i32")                # the host calls embed the integer tensors themselves (FrTensor::get_data)
    host.set_int_folds(not args.no_int_folds)   # ... except where an opening or an evaluation can fold the integers directly
    T, D, H, HD, F = args.seq, 4096, 32, 128, 11008
    FP = 16384                                  # rows of 11008 are padded to 16384 (src/tlookup.cu:301)
    SH = 16
    dev = "cuda"
    g = torch.Generator(device=dev)
    g.manual_seed(777)

    def gauss(*shape):
        x = torch.randn(*shape, generator=g, device=dev, dtype=torch.float32) * SIGMA
        return x.round().clamp_(-32768, 32767).to(torch.int32)

    weights = {"q": gauss(D, D), "k": gauss(D, D), "v": gauss(D, D), "o": gauss(D, D),
               "gate": gauss(F, D), "up": gauss(F, D), "down": gauss(D, F)}
    gens = ops.g1_make_generators(seeded_scalars(4096, SEED_G))
    table = ops.g1_table_gen(gens, 256)            # reference-format table handed to Hyrax
    NPTS = 4096
    fr_scale = _fr_const(1 << SH)[0]
    c_blind = rand_fr(1, 999)                      # the openings' blinding challenge (Fr c, test/llm.cu:52)
    seed = [1000]

    def chal(n):
        seed[0] += 1
        return rand_fr(n, seed[0])

    def log2c(n):
        return 0 if n <= 1 else (n - 1).bit_length()

    times = {"commit_weights": 0.0, "matmul": 0.0, "lookup": 0.0, "lookup_commits": 0.0, "open": 0.0}
    wall = {"commit_weights": 0.0, "remainder_blocks": 0.0, "matmul_blocks": 0.0, "mapping_blocks": 0.0, "io_openings": 0.0}
    counts = {"matmul": 0, "lookup": 0, "open": 0}

    class Block:
        """one timer block of the driver: wall clock between two device synchronisations"""
        def __init__(self, key):
            self.key = key

        def __enter__(self):
            torch.cuda.synchronize()
            self.t0 = time.perf_counter()

        def __exit__(self, *exc):
            torch.cuda.synchronize()
            wall[self.key] += time.perf_counter() - self.t0

    def require(ok, what):
        if not ok:
            raise SystemExit("bench.py layer: " + what)

    def pad_rows(flat_i32, rows, cols):
        """int tensor [rows][cols] -> [rows][16384] when cols is 11008, as the reference pads"""
        if cols == F:
            return ops.i32_pad(flat_i32, F, FP, rows * FP)
        return flat_i32

    def open_i32(flat_i32, point):
        """get_data + Hyrax::open (rows of 4096 columns); returns the opened evaluation"""
        n = flat_i32.numel()
        res = host.hyrax_open(flat_i32, n, 4096, table, NPTS, point, c_blind, com_scale=1)
        times["open"] += host.last_prove_seconds()
        counts["open"] += 1
        return res

    def commit_weight(w):
        flat = w.contiguous().view(-1)
        if w.shape[1] != 4096:                     # down: rows of 11008 padded to 16384
            flat = pad_rows(flat, w.shape[0], w.shape[1])
        n = flat.numel()
        with Block("commit_weights"):
            t0 = time.perf_counter()
            host.hyrax_commit_i32(flat, n, 4096, table, NPTS, com_scale=1)
            torch.cuda.synchronize()
            times["commit_weights"] += time.perf_counter() - t0

    def rescale(y):
        """y exact int64 -> (quotient int32, remainder int32) with y = q*2^16 + r, r in [-2^15, 2^15)"""
        q = (y + (1 << (SH - 1))) >> SH
        r = y - (q << SH)
        return q.to(torch.int32), r.to(torch.int32)

    def remainder_block(r, rows, cols, u):
        """test/llm.cu:98-108: the remainder's range lookup at the product's point and its opening, which must agree"""
        with Block("remainder_blocks"):
            flat = r.contiguous().view(-1)
            n = flat.numel()
            res = host.tlookup_range_prove(flat, n, -(1 << 15), 1 << 16, chal(1), chal(len(u)), u, table, NPTS, 1, 4096, want_m=False)
            times["lookup"] += host.last_prove_seconds()
            times["lookup_commits"] += res["commit_s"]
            counts["lookup"] += 1
            if os.environ.get("GRAPE_BENCH_VERBOSE"):
                print("  range lookup n=%d: %.4f s (commitments %.4f)" % (n, host.last_prove_seconds(), res["commit_s"]), file=sys.stderr)
            opened = open_i32(pad_rows(flat, rows, cols), u)
            require(np.array_equal(opened, res["S_claim"]), "a remainder's lookup value and its opening disagree")
        return res["S_claim"]

    # the two mapping lookup objects live as long as the prover (the reference's driver constructs them once, before its loop over
    # the layers, test/llm.cu:63-64), so each keeps the r drawn at its construction and the rows B[t]*G_i of its occupied entries
    mapping_r = {}
    mapping_stats = []

    def mapping_block(x_in, x_out, rows, cols, low, length, fmap):
        """test/llm.cu:152-164: the mapping lookup and the openings of its two tensors"""
        with Block("mapping_blocks"):
            a, b = x_in.contiguous().view(-1), x_out.contiguous().view(-1)
            n = a.numel()
            if (low, length) not in mapping_r:
                mapping_r[(low, length)] = chal(1)
            r = mapping_r[(low, length)]
            u = chal(log2c(n))
            res = host.tlookup_mapping_prove_ex(a, b, n, low, length, fmap, chal(1), r, chal(log2c(n)), u, table, NPTS, 1, 4096)
            times["lookup"] += host.last_prove_seconds()
            times["lookup_commits"] += host.last_commit_seconds()
            counts["lookup"] += 1
            mapping_stats.append({"elements": n, "table": length, "entries_with_a_row": res[3], "elements_as_full_width_scalars": res[4],
                                  "rows_kept_from_an_earlier_proof": bool(res[5])})
            if os.environ.get("GRAPE_BENCH_VERBOSE"):
                print("  mapping lookup n=%d len=%d: %.4f s (commitments %.4f; %d table entries with a row of B[t]*G_i%s, %d elements "
                      "as full-width scalars)" % (n, length, host.last_prove_seconds(), host.last_commit_seconds(), res[3],
                                                  " (rows kept from an earlier proof)" if res[5] else "", res[4]), file=sys.stderr)
            v_in, v_out = open_i32(pad_rows(a, rows, cols), u), open_i32(pad_rows(b, rows, cols), u)
            require(np.array_equal(res[1], host.fr_op(0, v_in, host.fr_op(2, r, v_out))), "a mapping lookup disagrees with its openings")

    def matmul_block(a_int, b_int, L, N, M, K, q, r_value, u, weight=None):
        """sumcheck for Y[l][n][m] = sum_k A[l][n][k] B[l][m][k] on the claim q(u)*2^16 + r(u) (test/llm.cu:85-95,
        :106, :111-125), then the opening of the weight at the reassembled point"""
        with Block("matmul_blocks"):
            Mp = 1 << log2c(M)
            qv = host.mle_eval(pad_rows(q.contiguous().view(-1), L * N, M), L * N * Mp, u)
            claim = host.fr_op(0, host.fr_op(2, qv, fr_scale), r_value)
            v = chal(log2c(K) + log2c(L))
            _, _, ac, bc = host.prove_matmul(a_int.contiguous().view(-1), b_int.contiguous().view(-1), L, N, M, K, u, v, claim)
            times["matmul"] += host.last_prove_seconds()
            counts["matmul"] += 1
            if weight is not None:                 # L = 1: the point of B is v | u[:log M] (ReassembleVectors)
                wp = np.concatenate([v, u[: log2c(M)]])
                wflat = pad_rows(weight.contiguous().view(-1), weight.shape[0], weight.shape[1])
                if wflat.numel() != 1 << log2c(wflat.numel()):      # 11008 rows: zero rows up to 16384
                    wflat = torch.cat([wflat, torch.zeros((1 << log2c(wflat.numel())) - wflat.numel(), dtype=torch.int32, device=dev)])
                require(np.array_equal(open_i32(wflat, wp), bc), "a weight's opening disagrees with its sumcheck")

    def mm(a, b):      # exact: every product sum stays below 2^53
        return torch.matmul(a.to(torch.float64), b.to(torch.float64).transpose(-1, -2)).to(torch.int64)

    native = args.witness == "native"

    def mmr(a, b):
        """quotient and remainder of a . b^T at scale 2^16: the library's integer kernel, or torch"""
        if native:
            return ops.wit_matmul_rescale(a.contiguous(), b.contiguous(), 1 << SH)
        return rescale(mm(a, b))

    def product(a, b, L, N, M, K, weight=None):
        """witness (outside the timers), then the remainder block and the matmul block at one point u"""
        q, r = mmr(a, b)
        u = chal(log2c(L) + log2c(N) + log2c(M))
        r_value = remainder_block(r, L * N, M, u)
        del r
        matmul_block(a, b, L, N, M, K, q, r_value, u, weight)
        return q

    # synthetic tables for the two mapping lookups (the reference's own table files are not in its tree)
    exp_low, exp_len = -(1 << 19), 1 << 20
    xs = torch.arange(exp_len, dtype=torch.float64) + exp_low
    exp_map = torch.round(4095.0 * torch.exp((xs - (exp_len // 2 - 1)) / float(1 << 16))).to(torch.int32).numpy()
    silu_low, silu_len = -(1 << 18), 1 << 19
    xs = (torch.arange(silu_len, dtype=torch.float64) + silu_low) / 1024.0
    silu_map = torch.round(1024.0 * xs * torch.sigmoid(xs)).to(torch.int32).numpy()
    d_exp_map, d_silu_map = torch.from_numpy(exp_map).cuda(), torch.from_numpy(silu_map).cuda()

    def one_layer(spread=False):
        for d in (times, wall):
            for k in d:
                d[k] = 0.0
        counts["matmul"] = counts["lookup"] = counts["open"] = 0
        del mapping_stats[:]
        x = gauss(T, D)                            # fresh activations for every layer
        for w in weights.values():
            commit_weight(w)
        with Block("io_openings"):                 # the block input's opening (test/llm.cu:604-608)
            open_i32(x.view(-1), chal(log2c(T * D)))
        # attention projections
        proj = {}
        for name in ("q", "k", "v"):
            proj[name] = product(x, weights[name], 1, T, D, D, weights[name])
        qh = proj["q"].view(T, H, HD).permute(1, 0, 2).contiguous()
        kh = proj["k"].view(T, H, HD).permute(1, 0, 2).contiguous()
        vh = proj["v"].view(T, H, HD).permute(1, 2, 0).contiguous()       # [H][HD][T]
        sc_q = product(qh, kh, H, T, T, HD)                                # [H][T][T]
        if spread:
            # the same layer with softmax scores spread uniformly over the exponential's table: no entry is occupied often
            # enough for a row of B[t]*G_i, so the logUp tensor is committed as full-width scalars
            e_in = torch.randint(exp_low, exp_low + exp_len, sc_q.shape, generator=g, device=dev, dtype=torch.int32)
        else:
            e_in = sc_q.clamp(exp_low, exp_low + exp_len - 1)
        del sc_q
        e_out = d_exp_map[(e_in - exp_low).long()]
        mapping_block(e_in, e_out, H * T, T, exp_low, exp_len, exp_map)
        del e_in
        av_q = product(e_out, vh, H, T, HD, T)                             # [H][T][HD]
        del e_out
        attn = av_q.permute(1, 0, 2).contiguous().view(T, D)
        x2 = product(attn, weights["o"], 1, T, D, D, weights["o"])
        # feed-forward
        gq = product(x2, weights["gate"], 1, T, F, D, weights["gate"])
        uq = product(x2, weights["up"], 1, T, F, D, weights["up"])
        s_in = gq.clamp(silu_low, silu_low + silu_len - 1)
        s_out = d_silu_map[(s_in - silu_low).long()]
        mapping_block(s_in, s_out, T, F, silu_low, silu_len, silu_map)
        hq, _ = rescale(s_out.to(torch.int64) * uq.to(torch.int64))
        dq = product(hq, weights["down"], 1, T, D, F, weights["down"])
        with Block("io_openings"):                 # the block output's opening (test/llm.cu:76-82)
            open_i32(dq.view(-1), chal(log2c(T * D)))
        return sum(wall.values())

    def snapshot(total):
        return {"value": float(total), "wall_breakdown_s": {k: float(v) for k, v in wall.items()},
                "provers_only_s": float(times["commit_weights"] + times["matmul"] + times["lookup"]),
                "provers_breakdown_s": {k: float(v) for k, v in times.items()},
                "mapping_lookups": [dict(m) for m in mapping_stats]}

    # the first layer of a process also builds the tables tied to the Hyrax object and to every
    # lookup object (wide fixed-base tables, B[t] * G_i); it is reported as the cold figure
    cold = None
    for i in range(args.warmup):
        t = one_layer()
        if i == 0:
            cold = snapshot(t)
    runs = []
    for _ in range(args.steps):
        runs.append(snapshot(one_layer()))
    total = float(np.mean([r["value"] for r in runs]))
    last = runs[-1]
    free_b, total_b = torch.cuda.mem_get_info()
    n_mm, n_lk, n_op = counts["matmul"], counts["lookup"], counts["open"]
    # the same layer on a witness that defeats the occupancy commitment (second of two such layers:
    # the first also replaces the rows kept from the layers above)
    spread = None
    if not args.no_spread:
        one_layer(spread=True)
        spread = snapshot(one_layer(spread=True))
    weight_points = sum(int(w.numel()) for w in weights.values())
    print(json.dumps({
        "metric": "layer_prove_time", "value": total, "unit": "s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": total * 1e3, "higher_is_better": False, "scaling": "weak", "vs_baseline": None, "dtype": "u32",
        "data": "synthetic",
        "config": {"workload": "configs[4]: LLaMA-2-7B-shape decoder layer proof, seq_len %d, d_model 4096, 32 heads x 128, "
                               "FFN 11008, int16 weights/activations" % T,
                   "scope": "wall clock of every proof block between two device synchronisations, as the reference's "
                            "total_prove_time (test/llm.cu:69-125): integer tensors -> Fr, copies, claim evaluation, sub-proof, "
                            "Hyrax openings; plus the 7 weight commitments; witness generation outside",
                   "integer_tensors": ("openings and claim evaluations fold their integer tensors directly (Hyrax::open(const int*), "
                                       "FrTensor::eval_ints) and the lookup provers index and embed their integer witnesses in one pass "
                                       "(tLookupRange::prove(const int*, ...), tLookupRangeMapping::prove(const int*, const int*, ...)): same "
                                       "proofs; prove_matmul(const int*, const int*, ...) folds the row variables of its operands from the integers") if not args.no_int_folds else
                                      "every integer tensor is embedded with FrTensor::get_data before its proof step (--no-int-folds)",
                   "wall_breakdown_s": last["wall_breakdown_s"],
                   "provers_only_s": float(np.mean([r["provers_only_s"] for r in runs])),
                   "provers_breakdown_s": last["provers_breakdown_s"],
                   "step_s": [r["value"] for r in runs],
                   "step_wall_breakdown_s": [r["wall_breakdown_s"] for r in runs],
                   "cold_s": cold["value"] if cold else None, "cold": cold,
                   "spread_s": spread["value"] if spread else None, "spread": spread,
                   "hbm_in_use_gib": (total_b - free_b) / 2**30, "hbm_total_gib": total_b / 2**30,
                   "mapping_lookups": last["mapping_lookups"],
                   "n_matmul_sumchecks": n_mm, "n_lookups": n_lk, "n_openings": n_op,
                   "weight_points": weight_points, "generators": NPTS,
                   "witness": "the library's integer kernels (grape_wit_matmul_rescale)" if native else "torch (float64 products, exact below 2^53)",
                   "note": "every layer draws fresh activations; Hyrax and lookup objects persist across layers as in the reference's "
                           "driver, so the tables tied to them are built by the first (cold) layer - the fixed-base tables, B[t]*G_i of "
                           "the range lookups, and the rows of the occupied entries of the two mapping lookups, which later layers "
                           "use again when their own witness sits on them (mapping_lookups); spread_s is the same layer with the "
                           "softmax scores uniform over the 2^20-entry table, where no such rows pay and the logUp tensor is "
                           "committed as full-width scalars; hbm_in_use_gib is what the process holds at the end "
                           "(tables, block cache, torch's pool)"}}))
    return 0


def matmul_workload(args):
    """Benchmark configuration configs[2]: prove_matmul of a 2048 x 4096 activation by a 4096 x 4096 weight
    (both int16-range, seeded), 12 sumcheck rounds over k after folding the row variables of both
    operands.  One step = one proof; the claim and the final evaluations are checked against
    independent multilinear evaluations on the GPU."""
    import torch
    from grape_amd import ops, _host as host
    from gpuutil import rand_fr
    ops.init(0)
    host.load()
    N, M, K = 2048, 4096, 4096
    dA = ops.fr_from_i32(torch.from_numpy(gaussian_i16((N, K), 31)).cuda())
    dB = ops.fr_from_i32(torch.from_numpy(gaussian_i16((M, K), 32)).cuda())
    u, v = rand_fr(23, 33), rand_fr(12, 34)
    du = ops.to_dev(u)
    a2, b2 = dA.clone(), dB.clone()
    ops.fr_fold(a2, N * K, du, N, 12, K)
    ops.fr_fold(b2, M * K, du, M, 0, K)
    claim = ops.fr_to_host(ops.fr_sum(ops.fr_mul(a2[:K].contiguous(), b2[:K].contiguous())))[0]
    del a2, b2
    secs = []
    for i in range(args.warmup + args.steps):
        _, _, ac, bc = host.prove_matmul(dA, dB, 1, N, M, K, u, v, claim)
        if i >= args.warmup:
            secs.append(host.last_prove_seconds())
    pa, pb = np.concatenate([v, u[12:23]]), np.concatenate([v, u[0:12]])
    if not (np.array_equal(host.mle_eval(dA, N * K, pa), ac) and np.array_equal(host.mle_eval(dB, M * K, pb), bc)):
        print("bench.py: final evaluations of prove_matmul differ from independent evaluations", file=sys.stderr)
        return 1
    t = float(np.mean(secs))
    print(json.dumps({
        "metric": "matmul_sumcheck_time", "value": t, "unit": "s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": t * 1e3, "higher_is_better": False, "scaling": "weak", "vs_baseline": None, "dtype": "u32",
        "data": "synthetic",
        "config": {"workload": "configs[2]: prove_matmul 2048x4096 by 4096x4096 (int16-range operands as Fr tensors)",
                   "operand_bytes": 32 * (N * K + M * K),
                   "operand_read_GBps": 32.0 * (N * K + M * K) / t / 1e9}}))
    return 0


def lookup_workload(args):
    """Benchmark configuration configs[3]: tLookupRange proof of 2^24 values in a 2^16-entry range with its
    commitments of A and m (4096 generators).  One step = one proof."""
    import torch
    from grape_amd import ops, _host as host
    from gpuutil import rand_fr
    import bigref as br
    ops.init(0)
    host.load()
    D, N, low = 1 << 24, 1 << 16, -32768
    S = np.random.default_rng(41).integers(low, low + N, size=D).astype(np.int32)
    gens = ops.g1_make_generators(rand_fr(4096, 42))
    table = ops.g1_table_gen(gens, 256)
    alpha, u, v = rand_fr(1, 43), rand_fr(24, 44), rand_fr(24, 45)
    secs, commits = [], []
    for i in range(args.warmup + args.steps):
        dS = ops.fr_from_i32(torch.from_numpy(S).cuda())
        res = host.tlookup_range_prove(dS, D, low, N, alpha, u, v, table, 4096, 1, 4096)
        if i >= args.warmup:
            secs.append(host.last_prove_seconds())
            commits.append(res["commit_s"])
    if br.fr_unpack(res["m"]) != [int(x) for x in np.bincount(S.astype(np.int64) - low, minlength=N)]:
        print("bench.py: multiplicities differ from numpy.bincount", file=sys.stderr)
        return 1
    t = float(np.mean(secs))
    print(json.dumps({
        "metric": "lookup_prove_time", "value": t, "unit": "s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": t * 1e3, "higher_is_better": False, "scaling": "weak", "vs_baseline": None, "dtype": "u32",
        "data": "synthetic",
        "config": {"workload": "configs[3]: tLookupRange, 2^24 lookups into a 2^16 range, 4096 generators",
                   "commit_s": float(np.mean(commits)),
                   "note": "tables tied to the Hyrax and lookup objects (fixed-base tables, B[t]*G_i) are built in the warm-up proof"}}))
    return 0


def claims_workload(args):
    """The two remaining sub-provers of the layer at its largest shapes: prove_eleMul on the gated
    feed-forward product (2048 rows of 11008 columns, padded to 16384: 2^25 index pairs, 25 rounds) and
    combine_claims of three claims on one 4096 x 4096 weight (24 rounds).  One step = one proof of each;
    the final evaluations are checked against independent multilinear evaluations on the GPU."""
    import torch
    from grape_amd import ops, _host as host
    from gpuutil import rand_fr
    ops.init(0)
    host.load()
    L, M, N, Np = 1, 2048, 11008, 16384
    rng = np.random.default_rng(61)
    dA = ops.fr_from_i32(torch.from_numpy(rng.integers(-(1 << 15), 1 << 15, M * N).astype(np.int32)).cuda())
    dB = ops.fr_from_i32(torch.from_numpy(rng.integers(-(1 << 15), 1 << 15, M * N).astype(np.int32)).cuda())
    u, v = rand_fr(25, 62), rand_fr(25, 63)
    zero = ops.to_dev(np.zeros((1, 4), dtype=np.uint64))
    pa, pb = ops.fr_pad(dA, N, Np, M * Np, zero), ops.fr_pad(dB, N, Np, M * Np, zero)
    claim = host.mle_eval(ops.fr_mul(pa, pb), M * Np, u)
    nv, num = 24, 3
    X = ops.fr_from_i32(torch.from_numpy(gaussian_i16((4096, 4096), 64)).cuda())
    us = np.stack([rand_fr(nv, 65 + j) for j in range(num)])
    vv = rand_fr(nv, 69)
    claims = np.stack([host.mle_eval(X, 1 << nv, us[j]) for j in range(num)])
    t_mul, t_comb = [], []
    for i in range(args.warmup + args.steps):
        _, _, ac, bc = host.prove_elemul(dA, dB, L, M, N, u, v, claim)
        t1 = host.last_prove_seconds()
        _, res = host.combine_claims(X, 1 << nv, claims, us, vv)
        t2 = host.last_prove_seconds()
        if i >= args.warmup:
            t_mul.append(t1)
            t_comb.append(t2)
    if not (np.array_equal(host.mle_eval(pa, M * Np, v), ac) and np.array_equal(host.mle_eval(pb, M * Np, v), bc)
            and np.array_equal(host.mle_eval(X, 1 << nv, vv), res)):
        print("bench.py: final evaluations differ from independent evaluations", file=sys.stderr)
        return 1
    t1, t2 = float(np.mean(t_mul)), float(np.mean(t_comb))
    print(json.dumps({
        "metric": "elemul_sumcheck_time", "value": t1, "unit": "s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": t1 * 1e3, "higher_is_better": False, "scaling": "weak", "vs_baseline": None, "dtype": "u32",
        "data": "synthetic",
        "config": {"workload": "prove_eleMul 2048 x 11008 (padded to 2^25 index pairs) and combine_claims of 3 claims on 2^24 elements",
                   "elemul_operand_read_GBps": 2 * 32.0 * M * N / t1 / 1e9,
                   "combine_claims_s": t2, "combine_claims_operand_read_GBps": 32.0 * (1 << nv) / t2 / 1e9}}))
    return 0


def mapping_workload(args):
    """The layer's largest single proof on its own: the softmax exponential's mapping lookup, 2^27 scores
    (32 heads x 2048 x 2048) into the 2^20-entry table, 4096 generators, scores distributed as the layer's
    are (Gaussian, sigma 181).  One step = one tLookupRangeMapping proof with its commitments of A and m;
    A goes through the table of the occupied entries (built by the warm-up proof and kept by the lookup
    object, as the reference's driver keeps its lookup objects across layers), or as full-width scalars
    with --plain-commit."""
    import torch
    from grape_amd import ops, _host as host
    from gpuutil import rand_fr
    ops.init(0)
    host.load()
    host.set_indexed_commit(not args.plain_commit)
    lg = args.log_elems if args.log_elems != 25 else 27
    D, N, low = 1 << lg, 1 << 20, -(1 << 19)
    exp_map, _ = host.witness_tables()
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    x = (torch.randn(D, generator=g, device="cuda") * 181.0).round().to(torch.int32).clamp_(low, low + N - 1)
    y = torch.from_numpy(exp_map).cuda()[(x - low).long()]
    gens = ops.g1_make_generators(rand_fr(4096, 42))
    table = ops.g1_table_gen(gens, 256)
    alpha, r, u, v = rand_fr(1, 43), rand_fr(1, 46), rand_fr(lg, 44), rand_fr(lg, 45)
    secs, commits = [], []
    for i in range(args.warmup + args.steps):
        res = host.tlookup_mapping_prove_ex(ops.fr_from_i32(x), ops.fr_from_i32(y), D, low, N, exp_map, alpha, r, u, v, table,
                                            4096, 1, 4096)
        if i >= args.warmup:
            secs.append(host.last_prove_seconds())
            commits.append(host.last_commit_seconds())
    t = float(np.mean(secs))
    print(json.dumps({
        "metric": "mapping_lookup_prove_time", "value": t, "unit": "s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": t * 1e3, "higher_is_better": False, "scaling": "weak", "vs_baseline": None, "dtype": "u32",
        "data": "synthetic",
        "config": {"workload": "tLookupRangeMapping, 2^%d lookups into the 2^20-entry exponential table, 4096 generators "
                               "(the softmax lookup of configs[4])" % lg,
                   "commit_s": float(np.mean(commits)),
                   "table_entries_with_a_row": res[3], "elements_as_full_width_scalars": res[4],
                   "rows_kept_from_an_earlier_proof": bool(res[5]),
                   "commit_of_A": "full-width scalars" if args.plain_commit else "table of the occupied entries, kept by the lookup object"}}))
    return 0


def witness_workload(args):
    """Witness generation for one LLaMA-2-7B-shape transformer block (d_model 4096, FFN 11008, one
    attention head as the reference's generator forces, seq_len 2048 by default): the C++
    LayerWitness class over the integer kernels.  One step = every tensor of the layer (quotients,
    remainders, softmax and SiLU table rows, RMSNorm parts).  Checks the proved relations on sampled
    entries, reports the matrix-product kernel against the measured multiply-add issue peak and the
    numpy oracle's exact integer product on a bounded sample of rows."""
    import torch
    from grape_amd import ops, _host as host
    ops.init(0)
    host.load()
    T, D, F = args.seq, 4096, 11008
    ops.wit_set_matmul_method({"auto": 0, "valu": 1, "mfma": 2}[args.matmul])
    g = torch.Generator(device="cuda")
    g.manual_seed(4242)

    def gauss(shape, sigma, clip=None):
        x = (torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * sigma).round()
        if clip:
            x = x.clamp_(-clip, clip - 1)
        return x.to(torch.int32)

    x = gauss((T, D), 65536.0)
    weights = {k: gauss(shape, SIGMA, 32768) for k, shape in (("Q", (D, D)), ("K", (D, D)), ("V", (D, D)), ("O", (D, D)),
                                                                ("gate", (F, D)), ("up", (F, D)), ("down", (D, F)))}
    weights["NormFirst"] = torch.full((D,), 65536, dtype=torch.int32, device="cuda")
    weights["NormSecond"] = torch.full((D,), 65536, dtype=torch.int32, device="cuda")
    e_np, s_np = host.witness_tables()
    d_exp, d_silu = torch.from_numpy(e_np).cuda(), torch.from_numpy(s_np).cuda()
    lw = host.LayerWitness(T, D, F)
    secs = []
    for i in range(args.warmup + args.steps):
        lw.generate(x, weights, d_exp, d_silu)
        if i >= args.warmup:
            secs.append(host.last_prove_seconds())
    t = float(np.mean(secs))

    # the relations the proofs rely on, on sampled entries of the full-size tensors
    rng = np.random.default_rng(3)
    S = 1 << 16
    n1 = lw.tensor("Q/normOutSecond").reshape(T, D).astype(np.int64)
    gate_w = weights["gate"].cpu().numpy().astype(np.int64)
    q, r = lw.tensor("Q/gate_out").reshape(T, F).astype(np.int64), lw.tensor("R/gate_out").reshape(T, F).astype(np.int64)
    for n, m in zip(rng.integers(0, T, 64).tolist(), rng.integers(0, F, 64).tolist()):
        if q[n, m] * (1 << 20) + r[n, m] != int(np.dot(n1[n], gate_w[m])):
            print("bench.py: gate projection witness is inconsistent", file=sys.stderr)
            return 1
    if r.min() < -(1 << 19) or r.max() >= (1 << 19):
        print("bench.py: remainder outside its range", file=sys.stderr)
        return 1
    out = lw.tensor("Q/output").astype(np.int64)
    if not np.array_equal(out, lw.tensor("Q/skip").astype(np.int64) + lw.tensor("Q/down_out").astype(np.int64)):
        print("bench.py: skip connection is inconsistent", file=sys.stderr)
        return 1
    del q, r, n1, out

    # dominant kernel: the gate/up projection's matrix product (T x 11008 x 4096), HIP events inside the library.
    # Activations below 2^22 take 3 signed byte planes, int16 weights 2: six int8 matrix-core products.
    h2 = torch.from_numpy(lw.tensor("Q/normOutSecond").reshape(T, D)).cuda()
    planes_a = 2 if int(h2.abs().max()) < (1 << 14) else 3
    planes_b = 2 if int(weights["gate"].abs().max()) < (1 << 14) else 3
    ops.profile_enable(True)
    ms = []
    for _ in range(6):
        ops.wit_matmul_rescale(h2, weights["gate"], 1 << 20)
        ms.append(ops.profile_last())
    ops.profile_enable(False)
    on_matrix_cores = len(ms[-1]) == 3      # plane split, the host's read of the operand magnitudes, the product
    kern_ms = float(np.median([m[-1] for m in ms[1:]]))
    split_ms = float(np.median([m[0] for m in ms[1:]])) if on_matrix_cores else 0.0
    mads = float(T) * D * F
    layer_mads = float(T) * D * (4 * D + 3 * F) + 2.0 * T * T * D
    if on_matrix_cores:
        int8_ops = 2.0 * planes_a * planes_b * mads
        # the library takes its 128 x 128 tile kernel when the product has a tile per CU
        kname = "wit_matmul_mfma_big_kernel" if ((T + 127) // 128) * ((F + 127) // 128) >= 256 else "wit_matmul_mfma_kernel"
        roofline = {"bound": "mfma", "kernel": "%s<%d,%d> (%d x %d x %d, int8 byte planes)" % (kname, planes_a, planes_b, T, F, D),
                    "achieved": int8_ops / (kern_ms * 1e-3) / 1e12, "peak": 5000.0, "unit": "TOP/s",
                    "frac": int8_ops / (kern_ms * 1e-3) / 1e12 / 5000.0, "traffic": None, "kernel_ms": kern_ms,
                    "plane_split_ms": split_ms,
                    "exact_multiplies_per_s": mads / ((kern_ms + split_ms) * 1e-3),
                    "note": "achieved counts the int8 operations the kernel executes (planes_a x planes_b products of the "
                            "exact 32-bit product); peak is the published dense int8 rate",
                    "layer_multiplies": layer_mads}
    else:
        peak = ops.bench_mad(16384, 512, 5)
        roofline = {"bound": "valu_int32_mul", "kernel": "wit_matmul_tiled_kernel (%d x %d x %d)" % (T, F, D),
                    "achieved": mads / (kern_ms * 1e-3) / 1e12, "peak": peak / 1e12, "unit": "Tmul/s",
                    "frac": mads / (kern_ms * 1e-3) / peak, "traffic": None, "kernel_ms": kern_ms,
                    "peak_source": "v_mad_u64_u32 issue-rate microbenchmark measured in this run",
                    "layer_multiplies": layer_mads}
    result = {
        "metric": "layer_witness_time", "value": t, "unit": "s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": t * 1e3, "higher_is_better": False, "scaling": "weak", "vs_baseline": None, "dtype": "int64",
        "data": "synthetic",
        "config": {"workload": "witness of one transformer block in the reference generator's fixed-point rules: seq_len %d, "
                               "d_model 4096, FFN 11008, one head; %d named int32 tensors" % (T, len(lw.names())),
                   "tensors": len(lw.names())},
        "roofline": roofline}
    if not args.no_cpu_baseline:
        from oracle import witness_oracle as wo
        rows = 512
        a = lw.tensor("Q/normOutSecond").reshape(T, D)[:rows]
        t0 = time.perf_counter()
        wq, wr = wo.rescale(wo.matmul_t(a, gate_w), 1 << 20)
        dt = time.perf_counter() - t0
        if not np.array_equal(wq, lw.tensor("Q/gate_out").reshape(T, F)[:rows]):
            print("bench.py: GPU and oracle quotients differ", file=sys.stderr)
            return 1
        result["cpu_baseline"] = {"value": rows * D * F / dt / 1e9, "unit": "Gmul/s", "cores": 1, "kind": "port",
                                  "sample": "first %d of %d rows of the gate projection (exact int64 numpy product), %.1f s" % (rows, T, dt),
                                  "gpu_same_unit": mads / ((kern_ms + split_ms) * 1e-3) / 1e9}
    lw.close()
    print(json.dumps(result))
    return 0


def rounds_workload(args):
    """The streaming kernels of the sumcheck and logUp rounds at 2^24 index pairs (tensors of 2^25
    elements, 1 GiB each, four times the Infinity Cache): the two-tensor round (src/prove.cu:29-46
    with its three reductions), the eq-weighted round with the fold fused in (element-product sumcheck
    and logUp rounds), the logUp sums alone, the MSB fold of two tensors and the element-wise product.
    Each is timed with events on the launch stream over `steps` launches; algorithmic bytes per index
    are the operands read once and the folded tensors written once.  One JSON line."""
    import torch
    from grape_amd import ops
    from gpuutil import rand_fr
    ops.init(0)
    lg = args.log_elems
    n, h = 1 << lg, 1 << (lg - 1)
    seeds = rand_fr(4, 77)
    v, beta = ops.to_dev(seeds[0:1]), ops.to_dev(seeds[1:2])
    A = ops.fr_from_i32(torch.arange(n, dtype=torch.int32, device="cuda"))
    B = ops.fr_from_i32(torch.arange(n, dtype=torch.int32, device="cuda") * 3 + 1)
    ops.fr_bcast_mul(A, ops.to_dev(seeds[2:3]), out=A)          # full-width values
    ops.fr_bcast_mul(B, ops.to_dev(seeds[3:4]), out=B)
    pyr = ops.eq_pyramid(ops.to_dev(rand_fr(lg - 1, 78)))
    e = pyr[h - 1: 2 * h - 1]

    def timed(fn):
        for _ in range(args.warmup):
            fn()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        e0.record()
        for _ in range(args.steps):
            fn()
        e1.record()
        torch.cuda.synchronize()
        return e0.elapsed_time(e1) / args.steps

    claim = ops.to_dev(rand_fr(1, 79))
    cases = [
        ("sumcheck2_kernel<two sums> + claim_final (grape_sumcheck_round2_claim, as prove_matmul's long rounds run)", 192, h,
         lambda: ops.sumcheck_round2_claim(A, B, n, h, v, claim)),
        ("sumcheck2_kernel<three sums> + final_sum (grape_sumcheck_round2)", 192, h, lambda: ops.sumcheck_round2(A, B, n, h, v)),
        ("wround2_kernel<beta, plain sums> + final (grape_wround2, logUp round)", 224, h,
         lambda: ops.wround2(A, B, beta, e, n, h, v, plain_sums=True)),
        ("wround2_kernel<beta, plain sums, inverse pair> + final (grape_wround2, first logUp round over A = 1/(S + beta))", 224, h,
         lambda: ops.wround2(A, B, beta, e, n, h, v, plain_sums=True, inverse_pair=True)),
        ("wround2_kernel<beta, plain sums, middle coefficient from the claim> + final (grape_wround2, long logUp rounds after the first)", 224, h,
         lambda: ops.wround2(A, B, beta, e, n, h, v, plain_sums=True, no_middle=True)),
        ("wround2_kernel<no beta> + final (grape_wround2, element-product round)", 224, h,
         lambda: ops.wround2(A, B, None, e, n, h, v)),
        ("tl_round_kernel + final_sum (grape_tlookup_round_sums, read only)", 160, h, lambda: ops.tlookup_round_sums(A, B, beta, e, h)),
        ("fold_msb_multi_kernel, two tensors", 192, h, lambda: ops.fr_fold_msb_multi([A, B], h, v)),
        ("ew_kernel<mul> (grape_fr_mul)", 96, n, lambda: ops.fr_mul(A, B, out=A)),
    ]
    out = []
    for name, bytes_per, units, fn in cases:
        ms = timed(fn)
        gbps = bytes_per * units / (ms * 1e-3) / 1e9
        out.append({"kernel": name, "bytes_per_unit": bytes_per, "units": units, "ms": ms, "GBps": gbps, "frac_of_hbm_peak": gbps / HBM_PEAK_GBPS})
    copy_ms = ops.bench_copy(1 << 30, 5)
    head = out[0]
    print(json.dumps({
        "metric": "round_kernel_bandwidth", "value": head["GBps"], "unit": "GB/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": head["ms"], "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "u32", "data": "synthetic",
        "config": {"workload": "sumcheck / logUp round kernels at 2^%d index pairs (tensors of 2^%d Fr elements)" % (lg - 1, lg)},
        "roofline": {"bound": "hbm", "achieved": head["GBps"], "peak": HBM_PEAK_GBPS, "unit": "GB/s", "frac": head["frac_of_hbm_peak"],
                     "traffic": None, "kernel": head["kernel"]},
        "kernels": out,
        "hbm_copy": {"kernel": "copy_kernel", "bytes_read": 1 << 30, "bytes_written": 1 << 30, "GBps": 2.0 * (1 << 30) / (copy_ms * 1e-3) / 1e9}}))
    return 0


def plumbing_workload(args):
    """Benchmark configuration configs[0] and the reduce-type kernels the other configurations lean on.
    2^16 seeded Fr elements times a second such tensor, the full sum of the product, and the
    Hyrax commitment of the product as a 256 x 256 matrix (256 MSMs of 256 full-width scalars) - checked
    against the CPU oracle, which is also timed.  Then, at sizes that stream from HBM: element-wise
    product, full sum, batched inversion (tlookup's A = 1/(S + beta)), the index + inverse-by-table pass
    of a lookup and its LDS-counted multiplicity histogram.  Every kernel is timed with events on the
    launch stream over `steps` launches; bytes per element are the operands read once and the result
    written once.  One JSON line."""
    import torch
    import orc
    from grape_amd import ops
    from gpuutil import rand_fr
    ops.init(0)

    def timed(fn, steps=None):
        steps = steps or args.steps
        for _ in range(args.warmup):
            fn()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        e0.record()
        for _ in range(steps):
            fn()
        e1.record()
        torch.cuda.synchronize()
        return e0.elapsed_time(e1) / steps

    # ---- configs[0]
    n0, side = 1 << 16, 256
    a, b = rand_fr(n0, 101), rand_fr(n0, 102)
    dA, dB = ops.to_dev(a), ops.to_dev(b)
    k = rand_fr(side, 103)
    gens = ops.g1_make_generators(k)
    c_bits = 13
    nw = (255 + c_bits - 1) // c_bits
    table = ops.g1_wide_table_gen(gens, c_bits, nw, 1 << (c_bits - 1))
    prod = ops.fr_mul(dA, dB)
    total = ops.fr_sum(prod)
    com = ops.commit_fr(prod, side, table, side, c_bits, nw, 1 << (c_bits - 1))
    t0 = time.perf_counter()
    h_prod = orc.vec2("orc_fr_vec_mul", a, b)
    h_sum = orc.fr_sum(h_prod)
    h_gens = orc.g1_make_generators(k)
    t1 = time.perf_counter()
    h_com = orc.commit_fr(h_prod, orc.g1_table(h_gens, 256), side, side)
    t2 = time.perf_counter()
    if not (np.array_equal(ops.fr_to_host(prod), h_prod) and np.array_equal(ops.fr_to_host(total)[0], h_sum)
            and np.array_equal(ops.g1_to_host(com), h_com)):
        print("bench.py: configs[0] differs from the CPU oracle", file=sys.stderr)
        return 1
    cfg0 = {
        "mul_ms": timed(lambda: ops.fr_mul(dA, dB, out=prod)),
        "sum_ms": timed(lambda: ops.fr_sum(prod)),
        "commit_ms": timed(lambda: ops.commit_fr(prod, side, table, side, c_bits, nw, 1 << (c_bits - 1), out=com)),
    }
    cfg0["commit_Mpoints_per_s"] = n0 / (cfg0["commit_ms"] * 1e-3) / 1e6
    cfg0["note"] = ("2^16 elements are launch-bound (4 MiB of operands); the commitment is 256 rows of 256 full-width scalars through "
                    "a %d-bit per-window table (%d additions per scalar)" % (c_bits, nw))
    cpu = {"value": n0 / (t2 - t1) / 1e6, "unit": "Mpoints/s", "cores": orc.lib().orc_num_threads(), "kind": "port",
           "sample": "the whole of configs[0]: 256 x 256 full-width commitment %.2f s (product, sum and generators %.3f s)" % (t2 - t1, t1 - t0)}
    del table

    # ---- streaming sizes
    lg = args.log_elems
    n = 1 << lg
    seeds = rand_fr(3, 104)
    X = ops.fr_from_i32(torch.arange(n, dtype=torch.int32, device="cuda") + 1)
    ops.fr_bcast_mul(X, ops.to_dev(seeds[0:1]), out=X)             # full-width, all non-zero
    Y = ops.fr_from_i32(torch.arange(n, dtype=torch.int32, device="cuda") * 5 + 3)
    ops.fr_bcast_mul(Y, ops.to_dev(seeds[1:2]), out=Y)
    out = ops.fr_empty(n)
    beta = ops.to_dev(seeds[2:3])
    lgw, tab_len, low = lg - 1, 1 << 16, -(1 << 15)
    nwit = 1 << lgw
    wit = torch.randint(low, low + tab_len, (nwit,), dtype=torch.int32, device="cuda")
    S = ops.fr_from_i32(wit)
    T, Btab = ops.tlookup_init(low, tab_len, ops.to_dev(rand_fr(1, 105)))
    idx1, A, mism = ops.tlookup_index_inverse(S, low, Btab)
    if mism != 0:
        print("bench.py: the witness is off its table", file=sys.stderr)
        return 1
    hist = torch.zeros(tab_len, dtype=torch.int32, device="cuda")
    cases = [
        ("ew_kernel<mul> (grape_fr_mul)", 96, n, lambda: ops.fr_mul(X, Y, out=out)),
        ("sum_kernel + final_sum (grape_fr_sum)", 32, n, lambda: ops.fr_sum(X)),
        ("inv_*_kernel, three-level batched inversion (grape_fr_shift_inverse, A = 1/(S + beta))", 64, n,
         lambda: ops.fr_shift_inverse(X, beta, out=out)),
        ("index_inverse_kernel (grape_tlookup_index_inverse: index, A = B[index])", 68, nwit,
         lambda: ops.tlookup_index_inverse(S, low, Btab)),
        ("hist_ranges + hist_lds<32768> + hist_merge (grape_tlookup_hist_index, 2^16 bins)", 4, nwit,
         lambda: ops.tlookup_hist_index(idx1, tab_len, hist=hist)),
    ]
    kernels = []
    for name, bytes_per, units, fn in cases:
        ms = timed(fn)
        gbps = bytes_per * units / (ms * 1e-3) / 1e9
        kernels.append({"kernel": name, "bytes_per_unit": bytes_per, "units": units, "ms": ms, "GBps": gbps,
                        "frac_of_hbm_peak": gbps / HBM_PEAK_GBPS, "units_per_s": units / (ms * 1e-3)})
    copy_ms = ops.bench_copy(1 << 30, 5)
    head = kernels[1]
    print(json.dumps({
        "metric": "fr_sum_bandwidth", "value": head["GBps"], "unit": "GB/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": head["ms"], "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "u32", "data": "synthetic",
        "config": {"workload": "configs[0] (2^16 Fr mul + sum + 256x256 Fr-path commit) and the reduce-type kernels at 2^%d elements "
                               "(lookup kernels at 2^%d)" % (lg, lgw),
                   "configs0": cfg0},
        "roofline": {"bound": "hbm", "achieved": head["GBps"], "peak": HBM_PEAK_GBPS, "unit": "GB/s", "frac": head["frac_of_hbm_peak"],
                     "traffic": None, "kernel": head["kernel"]},
        "kernels": kernels,
        "inversions_per_s": kernels[2]["units_per_s"],
        "cpu_baseline": cpu,
        "hbm_copy": {"kernel": "copy_kernel", "bytes_read": 1 << 30, "bytes_written": 1 << 30, "GBps": 2.0 * (1 << 30) / (copy_ms * 1e-3) / 1e9}}))
    return 0


def _fr_const(x):
    """Montgomery limbs of a small constant, as a (1, 4) uint64 array"""
    r = (21888242871839275222246405745257275088548364400416034343698204186575808495617 if CURVE == "bn254"
         else 0x73eda753299d7d483339d80809a1d80553bda402fffe5bfeffffffff00000001)
    v = (x << 256) % r
    return np.array([[(v >> (64 * i)) & ((1 << 64) - 1) for i in range(4)]], dtype=np.uint64)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=None)
    ap.add_argument("--warmup", type=int, default=None)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-pipelined", action="store_true",
                    help="commit workload: skip the second measurement (the same steps queued without waiting on three streams)")
    ap.add_argument("--no-spread", action="store_true",
                    help="layer workload: skip the two extra layers whose softmax scores are spread over the whole table")
    ap.add_argument("--no-int-folds", action="store_true",
                    help="layer workload: openings, claim evaluations and lookups embed their integer tensors first (FrTensor::get_data) "
                         "instead of reading the integers directly")
    ap.add_argument("--no-layer", action="store_true",
                    help="commit workload: skip the configs[4] layer proof that is measured afterwards in a child process")
    ap.add_argument("--log-elems", type=int, default=25, help="rounds workload: log2 of the tensors' element count")
    ap.add_argument("--workload", choices=["commit", "layer", "matmul", "lookup", "mapping", "witness", "rounds", "plumbing", "claims"], default="commit",
                    help="commit: configs[1], the metric's headline (default); matmul: configs[2]; "
                         "lookup: configs[3]; layer: configs[4]; mapping: the layer's softmax lookup on its own; "
                         "witness: the layer's witness generator; "
                         "rounds: the streaming kernels of the sumcheck / logUp rounds; "
                         "plumbing: configs[0] and the reduce-type kernels (sum, batched inversion, lookup index and histogram); "
                         "claims: prove_eleMul and combine_claims at the layer's largest shapes")
    ap.add_argument("--plain-commit", action="store_true",
                    help="mapping workload: commit A as full-width scalars instead of through its occupied entries")
    ap.add_argument("--seq", type=int, default=2048, help="sequence length of the layer and witness workloads")
    ap.add_argument("--matmul", choices=["auto", "valu", "mfma"], default="auto",
                    help="witness workload: integer matrix products on the matrix cores (auto, mfma) or with 64-bit multiply-adds (valu)")
    ap.add_argument("--witness", choices=["torch", "native"], default="native",
                    help="layer workload: who computes quotients and remainders of the matrix products")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py: this build runs the proving hot path on ONE GPU; --gpus %d is not supported "
              "(no collectives or sharding are part of it)" % args.gpus, file=sys.stderr)
        return 2
    if args.workload in ("rounds", "plumbing"):
        args.steps = 10 if args.steps is None else args.steps
        args.warmup = 2 if args.warmup is None else args.warmup
        return rounds_workload(args) if args.workload == "rounds" else plumbing_workload(args)
    if args.workload == "witness":
        args.steps = 3 if args.steps is None else args.steps
        args.warmup = 1 if args.warmup is None else args.warmup
        return witness_workload(args)
    if args.workload == "mapping":
        args.steps = 3 if args.steps is None else args.steps
        args.warmup = 1 if args.warmup is None else args.warmup
        return mapping_workload(args)
    if args.workload in ("matmul", "lookup", "claims"):
        args.steps = 5 if args.steps is None else args.steps
        args.warmup = 1 if args.warmup is None else args.warmup
        return {"matmul": matmul_workload, "lookup": lookup_workload, "claims": claims_workload}[args.workload](args)
    if args.workload == "layer":
        args.steps = 1 if args.steps is None else args.steps
        args.warmup = 1 if args.warmup is None else args.warmup
        return layer_workload(args)
    args.steps = 20 if args.steps is None else args.steps
    args.warmup = 3 if args.warmup is None else args.warmup

    import torch
    from grape_amd import ops
    ops.init(0)

    # ---- synthetic inputs, resident in HBM before the timed region
    W = gaussian_i16((ROWS, COLS), SEED_W)
    dW = torch.from_numpy(W).cuda()
    gens = ops.g1_make_generators(seeded_scalars(COLS, SEED_G))
    ops.sync()
    t0 = time.perf_counter()
    table = ops.g1_wide_table_gen(gens, RADIX_BITS, 1, K_DIGIT)
    ops.sync()
    table_gen_s = time.perf_counter() - t0
    out = ops.g1_empty(ROWS)
    points = ROWS * COLS

    def step():
        ops.commit_i32(dW, COLS, table, COLS, RADIX_BITS, 1, K_DIGIT, out=out)

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    ms_per_step = (time.perf_counter() - t0) * 1e3 / args.steps
    value = points / (ms_per_step * 1e-3) / 1e6
    # ---- dominant kernel, HIP events on the launch stream inside the library
    ops.profile_enable(True)
    kern_ms = []
    for _ in range(max(3, min(args.steps, 10))):
        step()
        kern_ms.append(ops.profile_last())
    ops.profile_enable(False)
    acc_ms = float(np.mean([k[0] for k in kern_ms]))
    red_ms = float(np.mean([k[1] for k in kern_ms]))
    peak_measured = ops.bench_mad(16384, 512, 5)
    achieved_alg = ALG_MULS_PER_POINT * points / (acc_ms * 1e-3)
    achieved_exec = EXEC_MULS_PER_POINT * points / (acc_ms * 1e-3)
    roofline = {
        "bound": "valu_int32_mul",
        "kernel": "commit_wide_kernel<int32>",
        # multiply-adds the kernel executes (one mixed addition per point), against the issue rate
        # of that instruction measured in this run
        "achieved": achieved_exec / 1e12,
        "peak": peak_measured / 1e12,
        "unit": "Tmul/s",
        "frac": achieved_exec / peak_measured,
        "mads_per_point": EXEC_MULS_PER_POINT,
        "points_per_launch": points,
        "traffic": COMMIT_KERNEL_TRAFFIC_BYTES if CURVE == "bls12_381" else None,
        "traffic_source": "recorded, not measured in this run: profiles/commit_wide_kernel_configs1_pmc_traffic.txt "
                          "(rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE of this command, scaled by the 1 GiB copy kernel; "
                          "FETCH_SIZE unit 2 KiB, WRITE_SIZE unit 1 KiB); algorithmic bytes 2.28e9",
        # the same launch priced as the reference's algorithm (two byte-window additions per int16
        # scalar): above the peak because the kernel does one addition per point, not two
        "reference_algorithm_equiv": {"muls_per_point": ALG_MULS_PER_POINT, "Tmul_per_s": achieved_alg / 1e12,
                                      "over_peak": achieved_alg / peak_measured},
        "frac_of_nominal_peak": achieved_exec / PEAK_MULS_NOMINAL,
        "peak_nominal": PEAK_MULS_NOMINAL / 1e12,
        "peak_source": "v_mad_u64_u32 issue-rate microbenchmark measured in this run "
                       "(no published integer-multiply peak exists for MI355X)",
        "kernel_ms": acc_ms,
        "reduce_kernel_ms": red_ms,
    }

    # ---- the same steps as a stream of independent commitments: queued without waiting
    # (grape_commit_i32_nowait) on three streams in turn, so that one commitment's row reduction - a
    # latency chain that occupies an eighth of the chip - runs under the next one's accumulation.
    # Every stream has its own output and its own digit-range flag, read at the end.  Measured after
    # the kernel timing above, which therefore sees the chip as the timed steps did.
    pipelined = None
    if not args.no_pipelined:
        n_streams = 3
        streams = [ops.stream_create() for _ in range(n_streams)]
        outs = [ops.g1_empty(ROWS) for _ in range(n_streams)]
        flags = torch.zeros(n_streams, dtype=torch.int32, device="cuda")

        def run(k):
            for i in range(k):
                j = i % n_streams
                ops.commit_i32_nowait(dW, COLS, table, COLS, RADIX_BITS, 1, K_DIGIT, outs[j], flags[j:j + 1], streams[j])
            for h in streams:
                ops.stream_sync(h)

        torch.cuda.synchronize()
        run(args.warmup)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        run(args.steps)
        torch.cuda.synchronize()
        pipe_ms = (time.perf_counter() - t0) * 1e3 / args.steps
        if int(flags.sum().item()) != 0:
            raise SystemExit("a queued commitment met a scalar outside the table's digits")
        for o in outs[:min(args.steps, n_streams)]:
            if not bool((o == out).all()):
                raise SystemExit("commitments queued on different streams differ from the one that was waited for")
        for h in streams:
            ops.stream_destroy(h)
        del outs
        pipelined = {"ms_per_step": pipe_ms, "value": points / (pipe_ms * 1e-3) / 1e6, "unit": "Mpoints/s", "streams": n_streams,
                     "note": "the same K steps as independent commitments queued without waiting on three streams in turn"}

    # ---- HBM side of the same kernel: one 128-byte table entry and one 4-byte scalar per point
    roofline["hbm_view"] = {"bytes_per_point": 132, "achieved_GBps": 132.0 * points / (acc_ms * 1e-3) / 1e9,
                            "peak_GBps": HBM_PEAK_GBPS, "frac": 132.0 * points / (acc_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS}

    # ---- plain copy of known size (the kernel the FETCH_SIZE / WRITE_SIZE counters are scaled by)
    copy_bytes = 1 << 30
    copy_ms = ops.bench_copy(copy_bytes, 5)
    hbm_copy = {"kernel": "copy_kernel", "bytes_read": copy_bytes, "bytes_written": copy_bytes,
                "GBps": 2.0 * copy_bytes / (copy_ms * 1e-3) / 1e9}

    # ---- the streaming Fr kernels: first fold pass over a 2^25-element tensor (1 GiB, reference
    # format, four times the Infinity Cache), duration from HIP events inside the library
    n_fold, c_fold = 1 << 25, 64
    t_fold = ops.fr_empty(n_fold)
    t_fold.zero_()
    x_fold = ops.to_dev(seeded_scalars(8, SEED_G + 1))
    ops.profile_enable(True)
    fold_ms = []
    torch.cuda.synchronize()
    for _ in range(6):
        # the tensor is all zero and stays so; it is not rewritten between runs, so no dirty
        # cache lines of a fill kernel are written back while the pass is timed
        ops.fr_fold(t_fold, n_fold, x_fold, c_fold, 0, n_fold // c_fold)
        fold_ms.append(ops.profile_last()[1])
    fold_ms = fold_ms[1:]
    ops.profile_enable(False)
    fold_pass_ms = float(np.median(fold_ms))
    fold_bytes = 32.0 * n_fold                                   # every element read once (writes: 1/32 more, not counted)
    roofline_streaming = {"bound": "hbm", "kernel": "fold_pass_kernel<1, false> (first pass of grape_fr_fold, c=64)",
                          "achieved": fold_bytes / (fold_pass_ms * 1e-3) / 1e9, "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                          "frac": fold_bytes / (fold_pass_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, "traffic": FOLD_KERNEL_TRAFFIC_BYTES,
                          "kernel_ms": fold_pass_ms, "elements": n_fold}
    del t_fold

    result = {
        "metric": "hyrax_commit_throughput",
        "value": value,
        "unit": "Mpoints/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "u32",
        "data": "synthetic",
        "config": {"workload": "configs[1]: Hyrax commit of a 4096x4096 int16-range matrix "
                               "(Gaussian sigma=2^10, clipped), 4096 seeded G1 generators, "
                               "small-scalar path, 4096 affine outputs",
                   "curve": CURVE, "rows": ROWS, "cols": COLS, "radix_bits": RADIX_BITS,
                   "table_bytes": int(table.numel()) * 4, "table_gen_s": table_gen_s},
        "roofline": roofline,
        "roofline_streaming": roofline_streaming,
        "hbm_copy": hbm_copy,
    }
    if pipelined:
        result["pipelined"] = pipelined

    if not args.no_cpu_baseline:
        base, cpu_out = cpu_baseline(W, gens, ops)
        got = ops.g1_to_host(out)[: cpu_out.shape[0]]
        if not np.array_equal(got, cpu_out):
            print("bench.py: GPU commitments differ from the CPU oracle on the sampled rows", file=sys.stderr)
            return 1
        result["cpu_baseline"] = base
    if not args.no_layer:
        # the metric's second figure: configs[4], measured by this same program in a child process
        # (its tables take most of the HBM, so this process first gives its own back)
        del table, dW, out
        torch.cuda.empty_cache()
        result["layer_prove_time"] = layer_in_child()
    print(json.dumps(result))
    return 0


def layer_in_child():
    """`bench.py --workload layer` (two warm-up layers - the cold one that builds the tables and one more, after which the
    block cache holds every size a layer asks for - and two timed) as a child process; returns its
    figures, or the reason why there are none - the commit figure above does not depend on it."""
    import subprocess
    cmd = [sys.executable, os.path.abspath(__file__), "--workload", "layer", "--steps", "2", "--warmup", "2"]
    try:
        res = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
        lines = [l for l in res.stdout.splitlines() if l.startswith("{")]
        if res.returncode != 0 or not lines:
            return {"value": None, "unit": "s", "error": (res.stderr or res.stdout)[-300:]}
        d = json.loads(lines[-1])
        c = d["config"]
        return {"value": d["value"], "unit": "s", "steps": d["steps"], "warmup": d["warmup"], "workload": c["workload"],
                "scope": c["scope"], "integer_tensors": c["integer_tensors"], "wall_breakdown_s": c["wall_breakdown_s"], "provers_only_s": c["provers_only_s"],
                "provers_breakdown_s": c["provers_breakdown_s"], "step_s": c["step_s"],
                "cold_s": c["cold_s"], "cold_wall_breakdown_s": c["cold"]["wall_breakdown_s"] if c["cold"] else None,
                "spread_s": c["spread_s"], "spread_wall_breakdown_s": c["spread"]["wall_breakdown_s"] if c["spread"] else None,
                "hbm_in_use_gib": c["hbm_in_use_gib"], "hbm_total_gib": c["hbm_total_gib"],
                "mapping_lookups": c["mapping_lookups"], "n_openings": c["n_openings"],
                "note": "value = a layer with the one-off tables in place, timed in the reference's total_prove_time scope; "
                        "provers_only_s = the sum of the provers' own timers; cold_s = the first layer of the process, which also "
                        "builds the tables; spread_s = the same layer with softmax scores uniform over the exponential's table"}
    except Exception as e:      # a time-out or a missing interpreter: report, do not fail the headline
        return {"value": None, "unit": "s", "error": str(e)[-300:]}


if __name__ == "__main__":
    sys.exit(main())
