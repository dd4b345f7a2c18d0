"""Folds and rounds that keep their operands, against the in-place forms."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from grape_amd import ops
    ops.init(0)
    return ops


# (outer, c, gap): nothing to bind, the finish kernel alone, one pass and several, with one outer index and many, ragged extents
@pytest.mark.parametrize("outer,c,gap", [(1, 1, 5), (3, 1, 7), (1, 2048, 1), (5, 100, 3), (1, 1 << 17, 1), (1, 11008, 16), (3, 5000, 40), (300, 16, 8),
                                         (300, 33, 100)])
def test_fold_of_a_kept_tensor(ops, outer, c, gap):
    from gpuutil import rand_fr
    from grape_amd import _capi
    N = outer * c * gap
    t = ops.to_dev(rand_fr(N, 701))
    x = ops.to_dev(rand_fr(20, 702))
    keep = t.clone()
    lib = _capi.load()
    out = torch.full((max(1, lib.grape_fr_fold_i32_elems(N, c, gap)), 8), -1, dtype=torch.int32, device="cuda")
    _capi.check(lib.grape_fr_fold_from(ops._p(out), ops._p(t), N, ops._p(x), c, 1, gap, ops._s()))
    assert torch.equal(t, keep)
    ops.fr_fold(t, N, x, c, 1, gap)
    assert torch.equal(out[: outer * gap], t[: outer * gap])


@pytest.mark.parametrize("in_size,n_out", [(2, 1), (600, 300), (1023, 512), (1 << 18, 1 << 17)])
def test_weighted_round_of_kept_operands(ops, in_size, n_out):
    from gpuutil import rand_fr
    A, S, E, v = (ops.to_dev(rand_fr(n, 710 + k)) for k, n in enumerate((in_size, in_size, n_out, 1)))
    a, s = A.clone(), S.clone()
    sums, Aw, Sw = ops.wround_kept(A, S, E, in_size, n_out, v)
    assert torch.equal(A, a) and torch.equal(S, s)
    want = ops.wround2(a, s, None, E, in_size, n_out, v)
    assert torch.equal(sums, want) and torch.equal(Aw, a[:n_out]) and torch.equal(Sw, s[:n_out])


@pytest.mark.parametrize("shift", [1, 2, 3])
def test_provers_take_operands_at_any_address(ops, shift):
    """views that start 4, 8 or 12 bytes behind a 16-byte boundary: the proofs of the same operands at a boundary"""
    from gpuutil import rand_fr
    from grape_amd import _host as host
    host.load()
    host.set_input_format("fr")

    def shifted(t):
        flat = torch.empty(t.numel() + shift, dtype=torch.int32, device="cuda")
        view = flat[shift:].view(t.shape)
        view.copy_(t)
        assert view.data_ptr() % 16 == 4 * shift
        return view

    n = 16
    a, b = ops.to_dev(rand_fr(n * n, 720)), ops.to_dev(rand_fr(n * n, 721))
    u, v = rand_fr(8, 722), rand_fr(8, 723)
    prod = ops.fr_mul(a, b)
    claim = host.mle_eval(prod, n * n, u)
    want = host.prove_elemul(a, b, 1, n, n, u, v, claim)
    for x, y in ((shifted(a), b), (a, shifted(b)), (shifted(a), shifted(b))):
        assert all(np.array_equal(p, q) for p, q in zip(want, host.prove_elemul(x, y, 1, n, n, u, v, claim)))
    # the matrix product's claim is what its proof over operands at a boundary accepts: sum_k A(u_row, k) B(u_col, k)
    x, y = a.clone(), b.clone()
    ops.fr_fold(x, n * n, ops.to_dev(u), n, 4, n)
    ops.fr_fold(y, n * n, ops.to_dev(u), n, 0, n)
    claim = ops.fr_to_host(ops.fr_sum(ops.fr_mul(x[:n].contiguous(), y[:n].contiguous())))[0]
    want = host.prove_matmul(a, b, 1, n, n, n, u, v[:4], claim)
    for x, y in ((shifted(a), b), (a, shifted(b))):
        assert all(np.array_equal(p, q) for p, q in zip(want, host.prove_matmul(x, y, 1, n, n, n, u, v[:4], claim)))
