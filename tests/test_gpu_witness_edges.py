"""Edges of the witness kernels' tiling: rows that are shorter than, equal to and longer than a workgroup's reach in the split into byte
planes, and table lookups of every alignment and tail."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from grape_amd import ops
    ops.init(0)
    return ops


# K: one padded step, a padded row, several rows a workgroup with threads left over (Kp = 320), exactly one group a thread (1024), a row that
# ends inside the first, the second and the last of the four groups in flight; more rows than workgroups at once
@pytest.mark.parametrize("N,M,K", [(1, 1, 4), (3, 5, 60), (33, 7, 64), (10, 70, 260), (5, 130, 1024), (3, 2, 1028), (2, 3, 2052), (4, 3, 4096), (2, 5, 4100),
                                   (9000, 2, 256), (2, 2100, 1000)])
def test_split_into_byte_planes(ops, N, M, K):
    from oracle import witness_oracle as wo
    rng = np.random.default_rng(N + M + K)
    a = rng.integers(-(1 << 21), 1 << 21, (N, K)).astype(np.int32)
    b = rng.integers(-(1 << 15), 1 << 15, (M, K)).astype(np.int32)
    a[-1, -1], b[-1, -1] = -(1 << 22) + 1, 1 << 16         # the magnitudes that choose the planes, at the very end
    ops.wit_set_matmul_method(2)
    try:
        q, r = ops.wit_matmul_rescale(torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), 1 << 31)
    finally:
        ops.wit_set_matmul_method(0)
    wq, wr = wo.rescale(wo.matmul_t(a, b), 1 << 31)
    assert np.array_equal(q.cpu().numpy(), wq) and np.array_equal(r.cpu().numpy(), wr)
    assert ops.wit_status() == 0


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 1024, 1025, 4099])
@pytest.mark.parametrize("offset", [0, 1, 4])
def test_table_lookup_alignments_and_tails(ops, n, offset):
    table = torch.randint(-(1 << 30), 1 << 30, (1000,), dtype=torch.int32, device="cuda")
    x = torch.randint(-500, 500, (n + offset,), dtype=torch.int32, device="cuda")[offset:]
    got = ops.wit_table_lookup(x, -500, table)
    assert torch.equal(got, table[(x + 500).long()]) and ops.wit_status() == 0
    for bad, k in ((-501, 0), (500, n - 1)):
        y = x.clone()
        y[k] = bad
        ops.wit_table_lookup(y, -500, table)
        assert ops.wit_status() == 2
