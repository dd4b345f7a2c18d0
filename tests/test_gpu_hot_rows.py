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
    new = np.nonzero(free & (want >= min_credit) & (h > 0))[0][:max_new]
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


def _steps(N, D, msm, proofs, room):
    """(rows, elements without one) that proofs of a witness spread evenly over N entries are committed with, (0, 0) where all of
    it goes the plain way: an entry is due once its elements have cost its row (23 additions a generator against 19 an element); a step
    costs a fifth of the commitment without rows (16 additions an element) and a quarter of what it saves by them (21 for each without
    a row where they are used), or what 2^17 elements without a row do, and twice that where half of a row's price comes back at once; rows are used from 30 % of the elements on; a
    step is made once due entries have had 2^17 elements since the last one"""
    each, row, due_at = D // N, 23.0 * msm, int(23.0 / 19.0 * msm) + 1
    held, credit, due, out = 0, 0, 0, []
    for i in range(proofs):
        cold = (N - held) * each
        credit += each
        if i > 0 and credit >= due_at:
            due += cold
            if due >= 1 << 17 and held < room:
                due = 0
                without = 16.0 * D
                now = min(21.0 * cold, without) if cold <= 0.7 * D else without
                spend = max(min(0.2 * without + 0.25 * (without - now), now), 19.0 * (1 << 17))
                new = min(int(spend / row), room - held, N - held)
                left = (N - held - new) * each
                if new == int(spend / row) and left <= 0.7 * D:
                    new = min(int(spend / (row - min(19.0 * each, row / 2))), room - held, N - held)
                held += new
                cold = (N - held) * each
        out.append((held, cold) if cold <= 0.7 * D else (0, 0))
    return out


def test_rows_grow_with_what_entries_have_cost(ops, host):
    """a witness spread evenly over 2^14 entries, 64 occurrences of each: no entry is worth a row of 64 in one proof, the object's
    second proof makes as many rows as a fifth of it pays for, the next ones more, in a table that has to be moved; they are used once
    they take in 30 %, and what is left is too little for a step of its own until several proofs have paid for it"""
    prove, low, N, D, msm = _prover(ops, host, 136, 14, 20, 900)
    rng = np.random.default_rng(901)
    even = [low + rng.permutation(np.arange(D, dtype=np.int64) % N) for _ in range(13)]
    even = [x.astype(np.int32) for x in even]
    want = _steps(N, D, msm, len(even), N)
    assert [n for n, _ in want[:3]] == [0, 0, 0] and 0 < want[3][0] < want[4][0] < N and want[10] == want[4] and want[11:] == [(N, 0)] * 2
    plain = [prove(x, indexed=False) for x in even]
    hot = []
    for i, x in enumerate(even):
        got = prove(x, fmt="i32" if i != 3 else "fr")
        _same(got, plain[i])
        hot.append(got[3:])
    assert [h[:2] for h in hot] == want
    assert [bool(h[2]) for h in hot] == [n > 0 for n, _ in want]


def _tight(ops, host, monkeypatch, seed):
    """2^16 entries and a budget whose eighth holds rows for half of them (BN254: 80 %): of 2 GiB the strided table over 257 generators takes
    0.88 and the per-window one over 64 columns 0.62 (BN254: 0.94 and 0.39), which leaves room for that eighth and a smaller table
    beside it that is moved there"""
    monkeypatch.setitem(os.environ, "GRAPE_TABLE_BUDGET_GIB", "2")
    prove, low, N, D, msm = _prover(ops, host, 257, 16, 20, seed)
    return prove, low, N, D, (2 << 30) // 8 // int(ops.init().grape_g1_wide_table_bytes(msm, 1, 1))


def test_rows_at_the_end_of_their_share(ops, host, monkeypatch):
    """2^16 entries that all come back: the rows stop growing at the end of their share, and those that are there stay: no others would
    take in more of the witness, however much the entries without a row have cost"""
    prove, low, N, D, share = _tight(ops, host, monkeypatch, 910)
    x = (low + np.random.default_rng(911).permutation(np.arange(D, dtype=np.int64) % N)).astype(np.int32)
    plain = prove(x, indexed=False)
    hot = []
    for _ in range(70):
        got = prove(x)
        _same(got, plain)
        hot.append(got[3])
    assert max(hot) == share < N and hot.index(share) < 30
    assert set(hot[hot.index(share):]) == {share}


def test_rows_of_another_witness(ops, host, monkeypatch):
    """a witness over one half of the entries until they have rows, then one over the other: once the share is taken, the rows that no
    element sits on are given up for those that have been missed"""
    prove, low, N, D, share = _tight(ops, host, monkeypatch, 915)
    rng = np.random.default_rng(916)
    for half in range(2):
        x = (low + half * N // 2 + rng.permutation(np.arange(D, dtype=np.int64) % (N // 2))).astype(np.int32)
        plain = prove(x, indexed=False)
        hot = []
        for _ in range(60):
            got = prove(x)
            _same(got, plain)
            hot.append(got[3:5])
            if got[3] >= N // 2 and got[4] == 0:
                break
        assert hot[-1][1] == 0 and N // 2 <= hot[-1][0] <= share
