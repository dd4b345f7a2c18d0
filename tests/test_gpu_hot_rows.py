"""Rows of a mapping lookup that grow over its proofs: entries get theirs once their elements have cost as much.  The kernels
against numpy; com(A) and the transcript of every proof against the plain full-width path."""
import ctypes
import os
import numpy as np
import pytest
import bigref as br
from gpuutil import rand_fr, assert_same

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from grape_amd import ops as o
    o.init(0)
    return o


@pytest.fixture(scope="module")
def host():
    from grape_amd import _host
    _host.load()
    return _host


# lengths around a tile (1024 entries) and a workgroup's share; counters that saturate; more due than there is room for
@pytest.mark.parametrize("n,min_credit,first,max_new", [(1, 5, 0, 8), (1023, 100, 3, 10 ** 6), (1025, 100, 0, 17), (5000, 1, 9, 400), (70001, 150, 70000, 70001)])
def test_credit_and_extension_kernels(ops, n, min_credit, first, max_new):
    import torch
    from grape_amd import _capi
    lib = ops.init()
    rng = np.random.default_rng(n)
    hist = (rng.integers(0, 200, n) * (rng.random(n) < 0.7)).astype(np.uint32)
    credit = rng.integers(0, 200, n).astype(np.uint32)
    credit[rng.random(n) < 0.05] = 0xffffffff - 50
    slot1 = np.where(rng.random(n) < 0.3, rng.integers(1, 1 + max(first, 1), n), 0).astype(np.int32)
    d = [torch.from_numpy(x.view(np.int32)).cuda() for x in (hist, credit, slot1)]
    p = [ctypes.c_void_p(x.data_ptr()) for x in d]
    info = (ctypes.c_uint64 * 3)()
    _capi.check(lib.grape_tlookup_hot_credit(p[0], n, p[2], p[1], min_credit, info, None))
    free = slot1 == 0
    want = np.where(free, np.minimum(credit.astype(np.int64) + hist, 0xffffffff), credit)
    assert np.array_equal(d[1].cpu().numpy().view(np.uint32), want.astype(np.uint32))
    h = hist.astype(np.int64)
    assert list(info) == [h[free].sum(), h[free & (want >= min_credit)].sum(), h[free & (h >= min_credit)].sum()]
    cold = (ctypes.c_uint64 * 1)()
    _capi.check(lib.grape_tlookup_hot_coverage(p[0], n, p[2], cold, None))
    assert cold[0] == info[0]
    lst = torch.zeros(n, dtype=torch.int32, device="cuda")
    given = (ctypes.c_uint64 * 2)()
    _capi.check(lib.grape_tlookup_hot_extend(p[0], p[1], n, min_credit, first, max_new, p[2], ctypes.c_void_p(lst.data_ptr()), given, None))
    new = np.nonzero(free & (want >= min_credit))[0][:max_new]
    slots = slot1.copy()
    slots[new] = first + 1 + np.arange(len(new))
    assert np.array_equal(d[2].cpu().numpy(), slots)
    assert np.array_equal(lst.cpu().numpy()[:len(new)], new)
    assert list(given) == [len(new), h[slots == 0].sum()]


# the host objects are found by their table's address: it stays taken until the process ends
_TABLES = []


def _prover(ops, host, npoints, logN, logD, seed):
    import torch
    low, N, D, msm = -(1 << (logN - 1)), 1 << logN, 1 << logD, 64
    fmap = np.random.default_rng(seed).integers(-1000, 1000, size=N).astype(np.int32)
    table = ops.g1_table_gen(ops.g1_make_generators(rand_fr(npoints, seed)), 256)
    _TABLES.append(table)
    alpha, r, u, v = rand_fr(1, seed + 1), rand_fr(1, seed + 2), rand_fr(logD, seed + 3), rand_fr(logD, seed + 4)

    def prove(s_in, indexed=True, fmt="i32"):
        host.set_indexed_commit(indexed)
        host.set_input_format(fmt)
        try:
            ins = [torch.from_numpy(x).cuda() for x in (s_in, fmap[s_in - low])]
            if fmt == "fr":
                ins = [ops.fr_from_i32(x) for x in ins]
            return host.tlookup_mapping_prove_ex(ins[0], ins[1], D, low, N, fmap, alpha, r, u, v, table, npoints, 1, msm)
        finally:
            host.set_indexed_commit(True)
            host.set_input_format("fr")
    return prove, low, N, D, msm


def _same(a, b):
    assert_same(a[0], b[0], "transcript")
    assert_same(a[1], b[1], "S(v)")
    assert_same(a[2], b[2], "com(A)")


def test_rows_grow_with_what_entries_have_cost(ops, host):
    """a witness spread evenly over 2^14 entries, 64 occurrences of each: no entry is worth a row of 64 in one proof, the object's
    third proof makes rows for as many as it pays for itself, the next for as many of the rest, in a table that has to be moved; what is
    left after it is too little for another step"""
    prove, low, N, D, msm = _prover(ops, host, 136, 14, 20, 900)
    rng = np.random.default_rng(901)
    even = [low + rng.permutation(np.arange(D, dtype=np.int64) % N) for _ in range(5)]
    even = [x.astype(np.int32) for x in even]
    each, due_at = D // N, int(1.8 * msm) + 1
    first = int(D * 19.0 / (23.0 * msm))
    second = first + int((N - first) * each * 19.0 / (23.0 * msm))
    assert 2 * each >= due_at > each and (N - first) * each >= 1 << 17 > (N - second) * each > 0
    plain = [prove(x, indexed=False) for x in even]
    hot = []
    for i, x in enumerate(even):
        got = prove(x, fmt="i32" if i != 3 else "fr")
        _same(got, plain[i])
        hot.append(got[3:])
    assert [h[0] for h in hot] == [0, 0, first, second, second]
    assert [h[1] for h in hot] == [0, 0] + [(N - n) * each for n in (first, second, second)]
    assert [bool(h[2]) for h in hot] == [False, False, False, True, True]


def test_rows_at_the_end_of_their_share(ops, host, monkeypatch):
    """2^16 entries that all come back, and a budget whose eighth holds a quarter of their rows: the rows stop growing there, and
    once what is missed has cost as much as they did they are given up for a new choice"""
    monkeypatch.setitem(os.environ, "GRAPE_TABLE_BUDGET_GIB", "1")
    # The per-window table takes what of the budget its windows fill: 24 x 1024 x 264 entries of 128 bytes (11-bit windows) are 0.77 GiB,
    # 22 x 2048 x 257 of 80 bytes (BN254, 12-bit windows) 0.86, and both leave the eighth that rows may take (264 generators of BN254
    # would leave 0.11 GiB).  Rows reach their share in the 10th and the 11th proof, and what is missed has then cost as much as
    # they did after four more at most.
    prove, low, N, D, msm = _prover(ops, host, 257 if br.CURVE == "bn254" else 264, 16, 20, 910)
    share = (1 << 30) // 8 // int(ops.init().grape_g1_wide_table_bytes(msm, 1, 1))
    x = (low + np.random.default_rng(911).permutation(np.arange(D, dtype=np.int64) % N)).astype(np.int32)
    plain = prove(x, indexed=False)
    hot = []
    for _ in range(18):
        got = prove(x)
        _same(got, plain)
        hot.append(got[3])
    assert max(hot) == share < N
    assert min(hot[hot.index(share):]) < share
