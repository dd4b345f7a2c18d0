"""Proofs whose long rounds carry their weights in a tensor, against the oracle's transcripts: the shortest that do, longer ones and
those that just do not, rows of odd length, points and challenges with coordinates 0 and 1, which have no inverse and take the rounds
that weigh every pair, and tables up to the witness's length with the commitments made beside the rounds."""
import numpy as np
import pytest

import bigref as br
import orc
from gpuutil import assert_same, rand_fr

pytestmark = pytest.mark.gpu

# (which of the two vectors, coordinate from the end, value): the first three rounds' factors, the last coordinate's own, a low variable
POINTS = [None, ("u", 1, 0), ("u", 1, 1), ("u", 2, 1), ("v", 1, 0), ("v", 1, 1), ("v", 2, 0), ("u", 17, 1)]


@pytest.fixture(scope="module")
def ops():
    from grape_amd import ops
    ops.init(0)
    return ops


# the host objects are found by their table's address: it stays taken until the process ends
_TABLES = []


@pytest.fixture(scope="module")
def table(ops):
    if not _TABLES:
        _TABLES.append(ops.g1_table_gen(ops.g1_make_generators(rand_fr(256, 915)), 256))
    return _TABLES[0]


@pytest.fixture(scope="module")
def host():
    from grape_amd import _host
    _host.load()
    yield _host
    _host.set_input_format("fr")


def _point(n, seed, special):
    u, v = rand_fr(n, seed), rand_fr(n, seed + 1)
    if special:
        name, back, value = special
        (u if name == "u" else v)[n - back] = br.fr_pack([value])[0]
    return u, v


@pytest.mark.parametrize("rows,cols,special", [(32, 1 << 16, s) for s in POINTS] + [(1 << 10, 3000, s) for s in (None, POINTS[1])] +
                         [(16, (1 << 17) + 1, None), (1, 1 << 21, None), (1 << 19, 5, None), (1 << 10, 2047, None), (1 << 13, 257, None), (1 << 14, 255, None)])
def test_element_product(ops, host, rows, cols, special):
    wide, n = 1 << (cols - 1).bit_length(), rows * cols
    A, B = rand_fr(n, 901), rand_fr(n, 902)
    u, v = _point((rows * wide).bit_length() - 1, 903, special)
    padded = np.zeros((rows, wide, 4), dtype=np.uint64)
    padded[:, :cols] = orc.vec2("orc_fr_vec_mul", A, B).reshape(rows, cols, 4)
    claim = orc.mle_eval(padded.reshape(-1, 4), u)
    st, transcript, last, at_a, at_b = orc.prove_elemul(A, B, 1, rows, cols, u, v, claim)
    assert st == 0
    host.set_input_format("fr")
    got = host.prove_elemul(ops.to_dev(A), ops.to_dev(B), 1, rows, cols, u, v, claim)
    for g, w, what in zip(got, (transcript, last, at_a, at_b), ("round polynomials", "final claim", "A(v)", "B(v)")):
        assert_same(g, w, what)
    with pytest.raises(host.HostError, match="claim != p\\(0\\) \\+ p\\(1\\)"):
        host.prove_elemul(ops.to_dev(A), ops.to_dev(B), 1, rows, cols, u, v, orc.fr_add(claim, br.fr_pack([1])[0]))


@pytest.mark.parametrize("logD,special", [(17, None), (18, None), (20, None)] + [(19, s) for s in POINTS])
def test_lookup(ops, host, table, logD, special):
    import torch
    D, N, low = 1 << logD, 1 << 6, -17
    rng = np.random.default_rng(logD)
    fmap = rng.integers(-1000, 1000, N).astype(np.int32)
    x = rng.integers(low, low + N, D).astype(np.int32)
    y = fmap[x - low]
    alpha, r = rand_fr(1, 911), rand_fr(1, 912)
    u, v = _point(logD, 913, special)
    beta = br.fr_pack([N])[0]
    host.set_input_format("i32")
    dx, dy = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    m = orc.tlookup_prep(orc.from_i32(x), low, N)
    S = orc.vec2("orc_fr_vec_add", orc.vec_bcast("orc_fr_vec_bcast_mul", orc.from_i32(y), r[0]), orc.from_i32(x))
    for mapping, s in ((False, orc.from_i32(x)), (True, S)):
        T, B = orc.tlookup_init(low, N, beta, *((orc.from_i32(fmap), r[0]) if mapping else ()))
        st, transcript, at_v = orc.tlookup_prove(s, T, B, m, alpha[0], beta, u, v)
        assert st == 0
        if mapping:
            got, claim = host.tlookup_mapping_prove(dx, dy, D, low, N, fmap, alpha, r, u, v, table, 256, 1, 256)
        else:
            res = host.tlookup_range_prove(dx, D, low, N, alpha, u, v, table, 256, 1, 256)
            got, claim = res["transcript"], res["S_claim"]
        assert_same(got, transcript, "transcript")
        assert_same(claim, at_v, "S(v)")


# a table that the caches hold beside a longer witness, one as long as the witness and one in between
@pytest.mark.parametrize("logD,logN", [(20, 12), (19, 17), (19, 19)])
@pytest.mark.parametrize("mapping", [False, True])
def test_lookup_and_its_commitments(ops, host, logD, logN, mapping):
    import torch
    gens, msm = 512, 256
    if len(_TABLES) < 2:
        _TABLES.append(ops.g1_table_gen(ops.g1_make_generators(rand_fr(gens, 916)), 256))
    table = _TABLES[1]
    htab = ops.g1_to_host(table)
    D, N, low = 1 << logD, 1 << logN, -(1 << (logN - 1))
    rng = np.random.default_rng(logD + logN)
    fmap = rng.integers(-30000, 30000, N).astype(np.int32)
    x = np.clip(np.round(rng.normal(0, N / 16, D)), low, low + N - 1).astype(np.int32)       # some entries often, many not at all
    x[:2] = low, low + N - 1
    y = fmap[x - low]
    alpha, r, u, v = rand_fr(1, 931), rand_fr(1, 932), rand_fr(logD, 933), rand_fr(logD, 934)
    beta = br.fr_pack([N])[0]
    S, m = orc.from_i32(x), orc.tlookup_prep(orc.from_i32(x), low, N)
    if mapping:
        S = orc.vec2("orc_fr_vec_add", orc.vec_bcast("orc_fr_vec_bcast_mul", orc.from_i32(y), r[0]), S)
    T, B = orc.tlookup_init(low, N, beta, *((orc.from_i32(fmap), r[0]) if mapping else ()))
    st, transcript, at_v = orc.tlookup_prove(S, T, B, m, alpha[0], beta, u, v)
    assert st == 0
    host.set_input_format("i32")
    dx, dy = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    for _ in range(2):                                   # the second proof finds the tables that the first one built
        if mapping:
            got, claim, com_A = host.tlookup_mapping_prove_ex(dx, dy, D, low, N, fmap, alpha, r, u, v, table, gens, 1, msm)[:3]
        else:
            res = host.tlookup_range_prove(dx, D, low, N, alpha, u, v, table, gens, 1, msm, want_commitments=True)
            got, claim, com_A = res["transcript"], res["S_claim"], res["com_A"]
            assert_same(res["m"], m, "m")
            mN = 1 << (logN // 2)
            for row in (0, N // mN // 2, N // mN - 1):
                assert_same(res["com_m"][row:row + 1], orc.commit_fr(m[row * mN:(row + 1) * mN], htab, mN, gens), "com(m) row %d" % row)
        assert_same(got, transcript, "transcript")
        assert_same(claim, at_v, "S(v)")
        for row in (0, D // msm // 3, D // msm - 1):
            A = B[x[row * msm:(row + 1) * msm] - low]
            assert_same(com_A[row:row + 1], orc.commit_fr(A, htab, msm, gens), "com(A) row %d" % row)
