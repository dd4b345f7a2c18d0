"""Lookups from their table indices alone: the index pass over integer witnesses (odd sizes, alignments, keys off the table),
the first round that gathers both tensors against the one that reads them, sparse commitments of table entries against those of
the tensor they make, and proofs whose witness misses the table."""
import ctypes
import numpy as np
import pytest
import torch
import bigref as br
import orc
from gpuutil import assert_same, rand_fr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from grape_amd import ops
    ops.init(0)
    return ops


@pytest.mark.parametrize("n", [1, 3, 4, 255, 1023, 1024, 4097, 70001])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("two", [False, True])
def test_index_pass_over_integers(ops, n, offset, two):
    from grape_amd import _capi
    rng = np.random.default_rng(n + offset)
    low, length = -37, 1 << 7
    table = rng.integers(-1000, 1000, length).astype(np.int32)
    key = rng.integers(low - 2, low + length + 2, n + offset).astype(np.int32)
    inside = (key >= low) & (key < low + length)
    second = table[np.clip(key - low, 0, length - 1)].copy()
    second[rng.random(n + offset) < 0.1] += 1
    bad = ~inside | ((second != table[np.clip(key - low, 0, length - 1)]) if two else False)
    dk, dc, dt = (torch.from_numpy(x).cuda() for x in (key, second, table))
    out = torch.full((n + 4,), -7, dtype=torch.int32, device="cuda")
    count = torch.empty(1, dtype=torch.int32, device="cuda")
    p = lambda t, skip=0: ctypes.c_void_p(t.data_ptr() + 4 * skip)
    rc = _capi.load().grape_tlookup_index_i32_nowait(p(out), p(dk, offset), p(dc, offset) if two else None, n, low, length, p(dt) if two else None,
                                                     p(count), None)
    assert rc == 0
    torch.cuda.synchronize()
    assert np.array_equal(out[:n].cpu().numpy(), np.where(inside, key - low + 1, 0)[offset:])
    assert (out[n:].cpu().numpy() == -7).all()
    assert int(count) == int(bad[offset:].sum())


@pytest.mark.parametrize("split", [False, True])
def test_first_round_gathers_both_tensors(ops, split):
    from grape_amd import _capi
    lib = _capi.load()
    n_out, length = 1 << 16, 1 << 10
    rng = np.random.default_rng(3)
    T = ops.to_dev(rand_fr(length, 11))
    beta, v = ops.to_dev(rand_fr(1, 12)), ops.to_dev(rand_fr(1, 13))
    B = ops.fr_shift_inverse(T, beta)
    idx = torch.from_numpy(rng.integers(1, length + 1, 2 * n_out).astype(np.int32)).cuda()
    S = T[idx.long() - 1].contiguous()
    A = B[idx.long() - 1].contiguous()
    u = ops.to_dev(rand_fr(16, 14))
    pyr = ops.eq_pyramid(u, 16)
    level = lambda j: pyr[(1 << j) - 1:(1 << (j + 1)) - 1].contiguous()
    tab = torch.empty(100, dtype=torch.int32, device="cuda")
    _capi.check(lib.grape_fold_tables(ctypes.c_void_p(tab.data_ptr()), ctypes.c_void_p(v.data_ptr()), 1, None))
    eq, high, period = level(16), None, 1
    if split:                                     # weights as products: the low variables' table and the high ones'
        period = 1 << 12
        eq, high = level(12), ops.eq_pyramid(u[12:].contiguous(), 4)[15:31].contiguous()
    p = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None
    out = []
    for gathered in (False, True):
        Ao, So = (ops.fr_empty(n_out) for _ in range(2))
        a = ops._Wround(A_out=p(Ao), S_out=p(So), A=p(A), S=p(S), idx1=p(idx) if gathered else None, B=p(B) if gathered else None, beta=p(beta), eq=p(eq),
                        eq_high=p(high), period=period, rowlen=1, rowpad=1, in_size=2 * n_out, n_out=n_out, v=p(v), plain_sums=2, tab=p(tab))
        if gathered:
            a.A = a.S = None
        partial = torch.empty(lib.grape_wround_partial_bytes(ctypes.byref(a)) // 4, dtype=torch.int32, device="cuda")
        a.partial = p(partial)
        sums = ops.fr_empty(5)
        if gathered:
            _capi.check(lib.grape_wround_queue_gathered(ctypes.byref(a), p(T), None))
        else:
            _capi.check(lib.grape_wround_queue(ctypes.byref(a), None))
        _capi.check(lib.grape_wround_finish(p(sums), 5, ctypes.byref(a), 1, None))
        out.append([x.cpu().numpy() for x in (sums, Ao, So)])
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("rows,live", [(5, 40), (5, 1), (4100, 3), (4097, 70), (64, 256)])
def test_sparse_commitment_of_table_entries(ops, rows, live):
    """`live` elements a row on average, a row without any among them; every share of the windows in a last batch, one and
    two rows a wave"""
    from grape_amd import _capi
    lib = _capi.load()
    cols, length, c = 256, 64, 10
    rng = np.random.default_rng(rows + live)
    gens = ops.g1_make_generators(rand_fr(cols, 21))
    table = ops.g1_wide_table_gen(gens, c, 26, 1 << (c - 1))
    entries = ops.to_dev(rand_fr(length, 22))
    idx = torch.from_numpy(rng.integers(1, length + 1, rows * cols).astype(np.int32)).cuda()
    skip = (rng.random((rows, cols)) >= live / cols).astype(np.int32)
    skip[rows // 2] = 1
    dskip = torch.from_numpy(skip.reshape(-1)).cuda()
    X = entries[idx.long() - 1].contiguous()
    plain = ops.commit_fr_sparse(X, dskip, cols, table, cols, c, 26, 1 << (c - 1))
    out = ops.g1_empty(rows)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    _capi.check(lib.grape_commit_fr_sparse_indexed(p(out), p(entries), p(idx), p(dskip), rows * cols, cols, p(table), cols, c, 26, 1 << (c - 1), None))
    assert torch.equal(out, plain)
    masked = X.clone()
    masked[dskip.bool()] = 0
    assert torch.equal(plain, ops.commit_fr(masked, cols, table, cols, c, 26, 1 << (c - 1)))
    J = 3
    nw = (255 + c - 1) // c
    nsets = (nw + J - 1) // J
    strided = ops.g1_strided_table_gen(gens, c, J, nsets)
    out2 = ops.g1_empty(rows)
    _capi.check(lib.grape_commit_fr_strided_masked_indexed(p(out2), p(entries), p(idx), p(dskip), rows * cols, cols, p(strided), cols, c, J, nsets, None))
    assert torch.equal(out2, plain)


_TABLES = []        # the host objects are found by their table's address: it stays taken until the process ends


# one long round, and long rounds that carry their weights
@pytest.mark.parametrize("logD", [17, 19])
@pytest.mark.parametrize("kind", ["range, key below", "range, key above", "mapping, key above", "mapping, wrong output"])
def test_proof_of_a_witness_off_its_table(ops, logD, kind):
    """one element off the table is refused; the object then proves a witness on it, refuses a point that is too short, and still
    refuses a padded witness of field elements that is off the table"""
    from grape_amd import _host as host
    host.load()
    if not _TABLES:
        _TABLES.append(ops.g1_table_gen(ops.g1_make_generators(rand_fr(256, 31)), 256))
    table = _TABLES[0]
    D, N, low, mapping = 1 << logD, 1 << 7, -40, kind.startswith("mapping")
    rng = np.random.default_rng(logD)
    fmap = rng.integers(-1000, 1000, N).astype(np.int32)
    alpha, r, u, v = rand_fr(1, 32), rand_fr(1, 33), rand_fr(logD, 34), rand_fr(logD, 35)
    beta = br.fr_pack([N])[0]
    T, B = orc.tlookup_init(low, N, beta, *((orc.from_i32(fmap), r[0]) if mapping else ()))

    def prove(x, y, fmt="i32", vars=logD):
        host.set_input_format(fmt)
        if fmt == "fr":
            dx, dy = (ops.to_dev(orc.from_i32(a)) for a in (x, y))
        else:
            dx, dy = (torch.from_numpy(a).cuda() for a in (x, y))
        try:
            if mapping:
                return host.tlookup_mapping_prove(dx, dy, x.size, low, N, fmap, alpha, r, u[:vars], v[:vars], table, 256, 1, 256)
            res = host.tlookup_range_prove(dx, x.size, low, N, alpha, u[:vars], v[:vars], table, 256, 1, 256)
            return res["transcript"], res["S_claim"]
        finally:
            host.set_input_format("fr")

    x = rng.integers(low, low + N, D).astype(np.int32)
    y = fmap[x - low]
    bad_x, bad_y = x.copy(), y.copy()
    if "output" in kind:
        bad_y[D // 3] += 1
    else:
        bad_x[D // 3] = low - 1 if "below" in kind else low + N
    with pytest.raises(host.HostError, match="claim != p\\(0\\) \\+ p\\(1\\)"):
        prove(bad_x, bad_y)
    S = orc.from_i32(x)
    if mapping:
        S = orc.vec2("orc_fr_vec_add", orc.vec_bcast("orc_fr_vec_bcast_mul", orc.from_i32(y), r[0]), S)
    st, transcript, at_v = orc.tlookup_prove(S, T, B, orc.tlookup_prep(orc.from_i32(x), low, N), alpha[0], beta, u, v)
    assert st == 0
    got, claim = prove(x, y)
    assert_same(got, transcript, "transcript")
    assert_same(claim, at_v, "S(v)")
    with pytest.raises(host.HostError, match="size"):
        prove(x, y, vars=logD - 1)
    n = D // 16384 * 11008                               # rows that the prover pads to 16384
    assert D // 3 < n
    x, y = bad_x[:n].copy(), bad_y[:n].copy()
    with pytest.raises(host.HostError, match="claim != p\\(0\\) \\+ p\\(1\\)"):
        prove(x, y, "fr")
