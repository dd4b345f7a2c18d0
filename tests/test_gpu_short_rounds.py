"""All short rounds of a sumcheck in one call (grape_short_rounds) against the same rounds one at a time: the entry points
that are compared with the oracle elsewhere.  Sizes around the elements of a workgroup (512), of a wave (64) and of a launch (nine
variables), rows that are no power of two, and the largest size accepted."""
import pytest
import torch

from gpuutil import rand_fr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from grape_amd import ops as o
    o.init(0)
    return o


def log2(n):
    return (n - 1).bit_length()


def sizes(size, row):
    while size > 1:
        out = size // 2 if size > row else 1 << (log2(size) - 1)
        yield size, out
        size = out


def same(ops, got, want, what):
    assert torch.equal(got.cpu(), want.cpu()), what


PAIRS = [(2, 2, 0), (3, 3, 0), (511, 511, 0), (513, 513, 0), (4096, 4096, 0), (11008, 11008, 0), (1 << 17, 1 << 17, 0),
         (2, 1, 1), (8 * 11008, 11008, 1), (1024 * 65, 65, 1), (1 << 16, 1 << 16, 1), (129, 129, 1), (512, 1, 1),
         (32 * 128, 128, 2), (4 * 300, 300, 2), (64, 1, 2), (2 * 65536, 65536, 2)]


@pytest.mark.parametrize("size,row,weights", PAIRS)
def test_pair_rounds(ops, size, row, weights):
    steps = list(sizes(size, row))
    A, B = ops.to_dev(rand_fr(size, 11)), ops.to_dev(rand_fr(size, 12))
    v = ops.to_dev(rand_fr(len(steps), 13))
    rows_log = log2(size // row)
    levels = len(steps) if weights == 1 else rows_log
    pyr = ops.eq_pyramid(ops.to_dev(rand_fr(max(levels, 1), 14)), max(levels - 1, 0))
    got, last = ops.short_rounds(0, [A, B], size, row, v, pyr if weights else None, max(levels - 1, 0), None, weights)
    for t, (n, out) in enumerate(steps):
        vt = v[len(steps) - 1 - t:len(steps) - t]
        lv = levels - 1 - t
        if weights == 1:
            rows = n > row
            want = ops.wround2(A, B, None, pyr[(1 << lv) - 1:], n, out, vt, rowlen=row if rows else 1, rowpad=1 << log2(row) if rows else 1)
        elif weights == 2 and n > row:
            want = ops.sumcheck_round2_seg(A, B, n, out, row, pyr[(1 << lv) - 1:], vt)
        else:
            want = ops.sumcheck_round2(A, B, n, out, vt)
        same(ops, got[t], want, "sums of round %d" % t)
    same(ops, last[0], A[0], "A")
    same(ops, last[1], B[0], "B")


@pytest.mark.parametrize("logn", [1, 2, 6, 7, 9, 10, 14, 16])
def test_lookup_rounds(ops, logn):
    n = 1 << logn
    beta, v = ops.to_dev(rand_fr(1, 20)), ops.to_dev(rand_fr(logn, 21))
    pyr = ops.eq_pyramid(ops.to_dev(rand_fr(logn, 22)), logn - 1)
    A, S, m = (ops.to_dev(rand_fr(n, 23 + k)) for k in range(3))
    got, last = ops.short_rounds(1, [A, S], n, n, v, pyr, logn - 1, beta, 1)
    table, table_last = ops.short_rounds(2, [A, S, m], n, n, v, pyr, logn - 1, beta, 1)
    A2, S2 = A.clone(), S.clone()
    for t in range(logn):
        half = n >> (t + 1)
        vt, e = v[logn - 1 - t:logn - t], pyr[half - 1:]
        same(ops, got[t], ops.wround2(A2, S2, beta, e, 2 * half, half, vt, plain_sums=True), "witness round %d" % t)
        same(ops, table[t], ops.tlookup_table_round(A, S, m, beta, e, half, vt), "table round %d" % t)
    same(ops, last[0], A2[0], "A")
    same(ops, last[1], S2[0], "S")
    same(ops, table_last[2], m[0], "m")


def test_refusals(ops):
    x = ops.to_dev(rand_fr(64, 30))
    v = ops.to_dev(rand_fr(8, 31))
    for args in ((0, [x, x], 1, 1, v), (0, [x, x], 63, 21, v), (1, [x, x], 64, 64, v), (0, [x, x], 1 << 18, 1 << 18, v)):
        with pytest.raises(Exception):
            ops.short_rounds(*args)
