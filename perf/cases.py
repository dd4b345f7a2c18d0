"""The work that a user of this framework has it do, as a list of measurable cases.

A prover commits to tensors (quantised weights, field tensors), proves matrix products, element-wise
products and table lookups about them, opens commitments and checks openings, and makes the integer
witness those proofs run on.  The sizes are those of a LLaMA-2-7B-shaped decoder layer (d_model 4096,
32 heads of 128, feed-forward width 11008, sequences of up to 2048) and of the small configurations,
and draw() spreads over the ranges in between.

Every result is a field element, a curve point or an integer, so it is compared exactly.
"""
import math

import numpy as np
import torch

from grape_amd import _host as host
from grape_amd import ops

GENERATORS = 4096          # columns of a committed row in a model: one set of generators for the prover's life
SMALL_GENERATORS = 256     # a small program's own set
SIGMA = 1024.0             # int16-range weights and activations

# 32 x 32 multiply-adds: one product of Fr, one mixed addition of a BLS12-381 point; a "flop" is half a multiply-add
FR_MUL = 2 * 136
G1_ADD = 2 * 3668

_public = {}


# ------------------------------------------------------------------ inputs
def _rng(seed):
    return np.random.default_rng(seed)


def _fr(rng, n):
    """n field elements as host words: residues below 2^254, all of them below the modulus"""
    x = rng.integers(0, 1 << 64, size=(n, 4), dtype=np.uint64)
    x[:, 3] &= np.uint64((1 << 62) - 1)
    return x


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _fr_dev(seed, n):
    """n full-width field elements on the GPU"""
    x = torch.randint(-(1 << 31), 1 << 31, (n, 8), generator=_gen(seed), device="cuda", dtype=torch.int32)
    x[:, 7] &= 0x3FFFFFFF
    return x


def _gauss(g, shape, sigma, limit):
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return x.mul_(sigma).round_().clamp_(-limit, limit - 1).to(torch.int32)


def _parameters(n):
    """The public parameters of a prover: n generators and their table, made once per program like its key files."""
    if n not in _public:
        ops.init(0)
        k = _fr(_rng(9000 + n), n)
        gens = ops.g1_make_generators(k)
        _public[n] = (gens, ops.g1_table_gen(gens, 256))
        torch.cuda.synchronize()
    return _public[n]


def _int16_table():
    """multiples of the generators, one signed 16-bit digit: what a program that commits int16 tensors keeps"""
    if "int16" not in _public:
        gens, _ = _parameters(GENERATORS)
        _public["int16"] = ops.g1_wide_table_gen(gens, 16, 1, 32768)
        torch.cuda.synchronize()
    return _public["int16"]


def _witness_tables():
    if "tables" not in _public:
        e, s = host.witness_tables()
        _public["tables"] = (e, s, torch.from_numpy(e).cuda(), torch.from_numpy(s).cuda())
    return _public["tables"]


def _log2(n):
    return max(0, (n - 1).bit_length())


def _words(a):
    """uint64 words of a host result as int64 (same bits)"""
    return np.ascontiguousarray(a).view(np.int64)


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # a product of two field tensors and its sum, the smallest piece of every protocol: latency and launches
        {"name": "fr_mul_sum_65536", "kind": "fr_mul_sum", "n": 65536},
        # prover and verifier of a small field tensor: commit 256 rows of 256, open at a point, check the opening
        {"name": "commit_open_verify_256x256", "kind": "open_verify", "rows": 256, "cols": 256},
        # the headline: row commitments of one quantised projection
        {"name": "commit_i32_4096x4096", "kind": "commit_i32", "rows": 4096, "cols": 4096},
        # a projection's product proved on field tensors
        {"name": "matmul_2048x4096x4096", "kind": "matmul", "L": 1, "N": 2048, "M": 4096, "K": 4096, "ints": False},
        # all heads' score products proved from the integer tensors
        {"name": "matmul_heads_i32", "kind": "matmul", "L": 32, "N": 2048, "M": 2048, "K": 128, "ints": True},
        # a short witness in a short range: the launches of a lookup proof
        {"name": "range_small", "kind": "range", "rows": 64, "cols": 256, "bits": 10, "ints": False},
        # the remainders of a rescaled product in their 2^16 range
        {"name": "range_i32_16777216", "kind": "range", "rows": 4096, "cols": 4096, "bits": 16, "ints": True},
        # SiLU: rows of 11008 padded to 16384, values spread as the witness generator spreads them
        {"name": "silu_2048x11008", "kind": "mapping", "rows": 2048, "cols": 11008, "table": "silu", "sigma": 4096.0},
        # the exponential of all heads' scores, the layer's largest proof: values concentrated on some entries
        {"name": "softmax_134217728", "kind": "mapping", "rows": 32768, "cols": 4096, "table": "exp", "sigma": 181.0},
        # the gated product of the feed-forward part, rows that are no power of two
        {"name": "elemul_2048x11008", "kind": "elemul", "rows": 2048, "cols": 11008},
        # the opening of a weight or remainder, one of two dozen in a layer
        {"name": "open_i32_4096x4096", "kind": "open", "rows": 4096, "cols": 4096, "ints": True},
        # every integer tensor of a layer
        {"name": "witness_2048", "kind": "witness", "seq": 2048, "dim": 4096, "hidden": 11008},
    ]


def _between(rng, lo, hi):
    """spread over the logarithm"""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _pow2(rng, lo, hi):
    return 1 << rng.randint(lo, hi)


def draw(rng):
    kind = rng.choice(["fr_mul_sum", "open_verify", "commit_i32", "matmul", "range", "mapping", "elemul", "open", "witness"])
    c = {"kind": kind}
    if kind == "fr_mul_sum":
        c["n"] = _between(rng, 256, 1 << 24)
    elif kind == "open_verify":
        c["rows"], c["cols"] = _pow2(rng, 2, 9), _pow2(rng, 4, 8)
    elif kind == "commit_i32":
        c["rows"], c["cols"] = _between(rng, 1, 8192), _between(rng, 64, 4096)
    elif kind == "matmul":
        # at most one extent of the product is no power of two, as in a model; the inner one is free
        c["L"] = rng.choice([1, 1, 4, 32])
        top = 4096 if c["L"] == 1 else 2048
        c["N"], c["M"] = _pow2(rng, 3, _log2(top)), _pow2(rng, 4, _log2(top))
        if c["L"] == 1 and rng.random() < 0.3:
            c["M"] = _between(rng, 64, 11008)
        c["K"] = _between(rng, 16, 11008 if c["L"] == 1 else 128)
        if c["L"] > 1:
            c["K"] = 1 << _log2(c["K"])
        c["ints"] = rng.random() < 0.5
    elif kind == "range":
        c["bits"] = rng.choice([8, 10, 12, 16])
        c["cols"] = _pow2(rng, 6, 12)
        low = max(1, c["bits"] - _log2(c["cols"]))
        c["rows"] = _pow2(rng, low, 25 - _log2(c["cols"]))
        c["ints"] = rng.random() < 0.5
        if rng.random() < 0.25:                          # rows of the feed-forward width, padded by the prover
            c["cols"], c["rows"], c["bits"] = 11008, _pow2(rng, 5, 11), 16
    elif kind == "mapping":
        c["table"] = rng.choice(["silu", "exp"])
        c["cols"] = _pow2(rng, 10, 12)
        c["rows"] = _pow2(rng, 21 - _log2(c["cols"]), 26 - _log2(c["cols"]))
        c["sigma"] = round(math.exp(rng.uniform(math.log(64.0), math.log(4096.0))), 1)
        if rng.random() < 0.4:
            c["cols"], c["rows"] = 11008, _pow2(rng, 7, 11)
        if c["rows"] * c["cols"] > (1 << 24):            # the largest spread no wider than a layer's
            c["sigma"] = round(min(c["sigma"], 1024.0), 1)
    elif kind == "elemul":
        c["rows"], c["cols"] = _pow2(rng, 3, 11), _between(rng, 64, 11008)
    elif kind == "open":
        c["rows"], c["cols"] = _pow2(rng, 2, 14), _pow2(rng, 6, 12)
        c["ints"] = rng.random() < 0.5
    else:
        c["seq"] = _between(rng, 32, 2048)
        c["dim"] = 128 * _between(rng, 2, 32)
        c["hidden"] = _between(rng, 512, 11008)
    return c


def _table_constant():
    """the constant r of a mapping lookup, drawn once for the life of the lookup object"""
    return _fr(_rng(77), 1)


def prepare(case, seed):
    ops.init(0)
    host.load()
    rng, kind = _rng(seed), case["kind"]
    st = dict(case)
    if kind == "fr_mul_sum":
        st["a"], st["b"] = _fr_dev(seed, case["n"]), _fr_dev(seed + 1000003, case["n"])
        return st
    if kind == "open_verify":
        n = case["rows"] * case["cols"]
        st.update(n=n, t=_fr_dev(seed, n), point=_fr(rng, _log2(n)), c=_fr(rng, 1), params=_parameters(SMALL_GENERATORS))
        return st
    if kind == "commit_i32":
        st.update(w=_gauss(_gen(seed), (case["rows"], case["cols"]), SIGMA, 32768), table=_int16_table())
        return st
    if kind == "matmul":
        return _prepare_matmul(st, case, seed, rng)
    if kind == "range":
        low, n = -(1 << (case["bits"] - 1)), case["rows"] * case["cols"]
        x = torch.randint(low, -low, (n,), generator=_gen(seed), device="cuda", dtype=torch.int32)
        nv = _log2(n)
        st.update(n=n, low=low, x=x if case["ints"] else ops.fr_from_i32(x), alpha=_fr(rng, 1), u=_fr(rng, nv), v=_fr(rng, nv),
                  msm=4096 if case["cols"] == 11008 else case["cols"], params=_parameters(GENERATORS))
        return st
    if kind == "mapping":
        exp, silu, d_exp, d_silu = _witness_tables()
        table, d_table = (exp, d_exp) if case["table"] == "exp" else (silu, d_silu)
        n, low = case["rows"] * case["cols"], -(table.shape[0] // 2)
        x = _gauss(_gen(seed), (n,), case["sigma"], -low)
        nv = _log2(n)
        st.update(n=n, low=low, x=x, y=d_table[(x - low).long()], table=table, alpha=_fr(rng, 1), u=_fr(rng, nv), v=_fr(rng, nv),
                  r=_table_constant(), msm=4096 if case["cols"] == 11008 else case["cols"], params=_parameters(GENERATORS))
        return st
    if kind == "elemul":
        return _prepare_elemul(st, case, seed, rng)
    if kind == "open":
        n = case["rows"] * case["cols"]
        w = _gauss(_gen(seed), (n,), SIGMA, 32768)
        st.update(n=n, t=w if case["ints"] else ops.fr_from_i32(w), point=_fr(rng, _log2(n)), c=_fr(rng, 1), params=_parameters(GENERATORS))
        return st
    # one layer's activations and weights at scale 2^16
    T, D, F = case["seq"], case["dim"], case["hidden"]
    g = _gen(seed)
    _, _, d_exp, d_silu = _witness_tables()
    shapes = {"Q": (D, D), "K": (D, D), "V": (D, D), "O": (D, D), "gate": (F, D), "up": (F, D), "down": (D, F)}
    weights = {k: _gauss(g, s, SIGMA, 32768) for k, s in shapes.items()}
    for k in ("NormFirst", "NormSecond"):
        weights[k] = torch.full((D,), 65536, dtype=torch.int32, device="cuda")
    st.update(x=_gauss(g, (T, D), 65536.0, 1 << 30), weights=weights, exp=d_exp, silu=d_silu, lw=host.LayerWitness(T, D, F))
    return st


def _prepare_matmul(st, case, seed, rng):
    L, N, M, K = case["L"], case["N"], case["M"], case["K"]
    g = _gen(seed)
    a, b = _gauss(g, (L * N * K,), SIGMA, 32768), _gauss(g, (L * M * K,), SIGMA, 32768)
    fa, fb = ops.fr_from_i32(a), ops.fr_from_i32(b)
    lu = _log2(L) + _log2(N) + _log2(M)
    u, v = _fr(rng, lu), _fr(rng, _log2(L) + _log2(K))
    du = ops.to_dev(u)
    x, y = fa.clone(), fb.clone()
    ops.fr_fold(x, L * N * K, du, N, _log2(M), K)
    ops.fr_fold(y, L * M * K, du, M, 0, K)
    prod = ops.fr_mul(x[: L * K].contiguous(), y[: L * K].contiguous())
    # the claim: the product's multilinear extension at u - sums over k, then the batch variables
    s = torch.cat([ops.fr_sum(prod[i * K:(i + 1) * K].contiguous()) for i in range(L)])
    host.set_input_format("fr")
    claim = host.mle_eval(s, L, u[lu - _log2(L):]) if L > 1 else ops.fr_to_host(s)[0]
    st.update(a=a if case["ints"] else fa, b=b if case["ints"] else fb, u=u, v=v, claim=claim)
    return st


def _prepare_elemul(st, case, seed, rng):
    rows, cols = case["rows"], case["cols"]
    g = _gen(seed)
    a, b = (ops.fr_from_i32(torch.randint(-(1 << 15), 1 << 15, (rows * cols,), generator=g, device="cuda", dtype=torch.int32)) for _ in range(2))
    wide = 1 << _log2(cols)
    nv = _log2(rows) + _log2(cols)
    u, v = _fr(rng, nv), _fr(rng, nv)
    prod = ops.fr_mul(a, b)
    if wide != cols:
        prod = ops.fr_pad(prod, cols, wide, rows * wide, ops.to_dev(np.zeros((1, 4), dtype=np.uint64)))
    host.set_input_format("fr")
    st.update(a=a, b=b, u=u, v=v, claim=host.mle_eval(prod, rows * wide, u))
    return st


class _View:
    """device memory of the witness object as a tensor"""

    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<i4", "data": (ptr, False), "version": 2}


def run(st):
    kind = st["kind"]
    if kind == "fr_mul_sum":
        p = ops.fr_mul(st["a"], st["b"])
        return p, ops.fr_sum(p)
    if kind == "commit_i32":
        return ops.commit_i32(st["w"], st["cols"], st["table"], GENERATORS, 16, 1, 32768)
    if kind == "witness":
        st["lw"].generate(st["x"], st["weights"], st["exp"], st["silu"])
        if "views" not in st:                            # the object's own buffers, the same from call to call
            st["views"] = {n: torch.as_tensor(_View(*st["lw"].device_ptr(n)), device="cuda") for n in st["lw"].names() if n[0] != "W"}
        return st["views"]
    host.set_input_format("i32" if st.get("ints", kind == "mapping") else "fr")
    if kind == "open_verify":
        res, ok = host.hyrax_open_verify(st["t"], st["n"], st["cols"], st["params"][1], SMALL_GENERATORS, st["point"], st["c"], com_scale=1)
        return _words(res), ok
    if kind == "open":
        return _words(host.hyrax_open(st["t"], st["n"], st["cols"], st["params"][1], GENERATORS, st["point"], st["c"], com_scale=1))
    if kind == "matmul":
        out = host.prove_matmul(st["a"], st["b"], st["L"], st["N"], st["M"], st["K"], st["u"], st["v"], st["claim"])
        return [_words(x) for x in out]
    if kind == "elemul":
        out = host.prove_elemul(st["a"], st["b"], 1, st["rows"], st["cols"], st["u"], st["v"], st["claim"])
        return [_words(x) for x in out]
    if kind == "range":
        r = host.tlookup_range_prove(st["x"], st["n"], st["low"], 1 << st["bits"], st["alpha"], st["u"], st["v"], st["params"][1], GENERATORS,
                                     1, st["msm"], want_commitments=True)
        return [_words(r[k]) for k in ("m", "transcript", "S_claim", "com_A", "com_m")]
    r = host.tlookup_mapping_prove_ex(st["x"], st["y"], st["n"], st["low"], st["table"].shape[0], st["table"], st["alpha"], st["r"], st["u"],
                                      st["v"], st["params"][1], GENERATORS, 1, st["msm"])
    return [_words(r[k]) for k in (0, 1, 2)]


def work(case):
    """Bytes: inputs once, outputs once.  Flops: two for a 32 x 32 multiply-add of the field and curve arithmetic that the
    protocols prescribe (one addition per int16 element or table entry committed, sixteen per full-width scalar)."""
    kind = case["kind"]
    if kind == "fr_mul_sum":
        return {"bytes": 96.0 * case["n"], "flops": float(FR_MUL) * case["n"]}
    if kind == "witness":
        T, D, F = case["seq"], case["dim"], case["hidden"]
        out = 23 * T * D + 6 * T * T + 7 * T * F
        return {"bytes": 4.0 * (4 * D * D + 3 * D * F + T * D + out), "flops": 2.0 * (T * D * (4.0 * D + 3.0 * F) + 2.0 * T * T * D)}
    if kind == "matmul":
        n = case["L"] * case["K"] * (case["N"] + case["M"])
        return {"bytes": (4.0 if case["ints"] else 32.0) * n, "flops": (40.0 if case["ints"] else FR_MUL) * n}
    n, rows = case["rows"] * case["cols"], case["rows"]
    if kind == "commit_i32":
        return {"bytes": 4.0 * n + 96.0 * rows + 96.0 * case["cols"], "flops": float(G1_ADD) * n}
    if kind == "open_verify":
        return {"bytes": 32.0 * n + 96.0 * (rows + case["cols"]), "flops": 16.0 * G1_ADD * n}
    if kind == "open":
        return {"bytes": (4.0 if case["ints"] else 32.0) * n, "flops": (40.0 if case["ints"] else FR_MUL) * n}
    if kind == "elemul":
        return {"bytes": 64.0 * n, "flops": 7.0 * FR_MUL * n}
    full = 1 << _log2(n)
    if kind == "range":
        return {"bytes": (4.0 if case["ints"] else 32.0) * n + 96.0 * full / min(4096, case["cols"]), "flops": (G1_ADD + 6.0 * FR_MUL) * full}
    return {"bytes": 8.0 * n + 96.0 * full / min(4096, case["cols"]), "flops": (G1_ADD + 6.0 * FR_MUL) * full}


def tolerance(case):
    return "exact"
