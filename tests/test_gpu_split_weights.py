"""Weighted rounds whose weight is a product of two tables' entries, against the round over the whole table of weights; rounds that
are finished together against rounds finished one by one; proofs on both sides of the longest prefix table."""
import ctypes

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from grape_amd import ops
    ops.init(0)
    return ops


def _weights(ops, period, n_out):
    from gpuutil import rand_fr
    rows = -(-n_out // period)
    low, high = ops.to_dev(rand_fr(period, 801)), ops.to_dev(rand_fr(rows, 802))
    full = ops.fr_mul(low.repeat(rows, 1), high.repeat_interleave(period, 0))[:n_out].contiguous()
    return low, high, full


# (period, in_size, n_out): one index a period, ragged rows, a last period that is cut off, an odd last pair, one period in all, a period
# that needs more workgroups than the smallest grid, threads of a wave in two periods, 24 and 1 periods a thread
CASES = [(1, 1 << 17, 1 << 16), (11008, 2 * 8 * 11008, 8 * 11008), (1000, 2 * 70001, 70001), (1 << 17, (1 << 18) - 1, 1 << 17), (100, 140001, 70001),
         (300000, 2 * 300000, 300000), (1 << 17, 1 << 22, 1 << 21), (4097, 2 * 4097 * 1537, 4097 * 1537)]


@pytest.mark.parametrize("period,in_size,n_out,mode", [c + (m,) for c in CASES for m in (0, 2, 3) if m != 2 or c[1] == 2 * c[2]])
def test_product_weights(ops, period, in_size, n_out, mode):
    from gpuutil import rand_fr
    A, S, v, beta = (ops.to_dev(rand_fr(n, 810 + k)) for k, n in enumerate((in_size, in_size, 1, 1)))
    beta = beta if mode else None
    low, high, full = _weights(ops, period, n_out)
    a, s = A.clone(), S.clone()
    got = ops.wround_products(A, S, beta, low, high, period, in_size, n_out, v, mode)
    want = ops.wround2(a, s, beta, full, in_size, n_out, v, plain_sums=mode != 0, inverse_pair=mode == 2, no_middle=mode == 3)
    assert torch.equal(got, want) and torch.equal(A[:n_out], a[:n_out]) and torch.equal(S[:n_out], s[:n_out])


@pytest.mark.parametrize("n_out", [1 << 16, 1 << 20])
def test_product_weights_of_a_gathered_tensor(ops, n_out):
    from gpuutil import rand_fr
    S, B, v, beta = (ops.to_dev(rand_fr(n, 820 + k)) for k, n in enumerate((2 * n_out, 1000, 1, 1)))
    idx1 = torch.randint(1, 1001, (2 * n_out,), dtype=torch.int32, device="cuda")
    low, high, full = _weights(ops, 1 << 14, n_out)
    s, A = S.clone(), ops.fr_empty(n_out)
    got = ops.wround_products(A, S, beta, low, high, 1 << 14, 2 * n_out, n_out, v, 2, idx1, B)
    want, a = ops.wround2_first_indexed(s, idx1, B, beta, full, n_out, v)
    assert torch.equal(got, want) and torch.equal(A, a) and torch.equal(S[:n_out], s[:n_out])


def test_refused_forms(ops):
    from grape_amd import _capi
    A, S, v, beta = ops.fr_empty(1 << 17), ops.fr_empty(1 << 17), ops.fr_empty(1), ops.fr_empty(1)
    low, high = ops.fr_empty(64), ops.fr_empty(1 << 10)
    for mode, b in ((1, beta), (0, beta), (2, None), (3, None)):
        with pytest.raises(_capi.GrapeError):
            ops.wround_products(A, S, b, low, high, 64, 1 << 17, 1 << 16, v, mode)
    lib = _capi.load()
    a = ops._Wround(n_out=1 << 16, eq_high=high.data_ptr(), period=0)
    assert lib.grape_wround_partial_bytes(ctypes.byref(a)) == 0


@pytest.mark.parametrize("rows,cols", [(2, 1 << 16), (4, 1 << 20), (1 << 9, 11008), (1 << 8, 5000), (2, 131073), (8, (1 << 18) + 5), (2, (1 << 20) + 1)])
def test_element_products_over_long_rows(ops, rows, cols):
    """the proof's own checks hold for the claim <eq(u), a b>, and the values left are the tensors' at v"""
    import numpy as np
    from gpuutil import rand_fr
    from grape_amd import _host as host
    n, lg = rows * cols, (rows - 1).bit_length() + (cols - 1).bit_length()
    wide = 1 << (cols - 1).bit_length()
    a, b = ops.to_dev(rand_fr(n, 830)), ops.to_dev(rand_fr(n, 831))
    u, v = rand_fr(lg, 832), rand_fr(lg, 833)
    zero = ops.to_dev(np.zeros((1, 4), dtype=np.uint64))
    pad = (lambda t: t) if wide == cols else (lambda t: ops.fr_pad(t, cols, wide, rows * wide, zero))
    host.set_input_format("fr")
    claim = host.mle_eval(pad(ops.fr_mul(a, b)), rows * wide, u)
    _, _, at_a, at_b = host.prove_elemul(a, b, 1, rows, cols, u, v, claim)
    for got, t in ((at_a, a), (at_b, b)):
        assert np.array_equal(got.reshape(-1), np.asarray(host.mle_eval(pad(t).clone(), rows * wide, v)).reshape(-1))
