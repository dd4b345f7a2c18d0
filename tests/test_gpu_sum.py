"""Sums of field tensors at the sizes where the launch changes (one workgroup, several, the most there are, remainders of a thread's
terms), again and again over the same counter, and two streams side by side."""
import numpy as np
import pytest
import orc
from gpuutil import rand_fr, assert_same

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from grape_amd import ops
    ops.init(0)
    return ops


@pytest.mark.parametrize("n", [1, 255, 256, 1024, 1025, 2048, 3000, 65536, 65537, 1 << 17, (1 << 17) + 1, 190003, 1 << 19, (1 << 19) + 1, (1 << 21) - 1, (1 << 21) + 1, (1 << 22) + 4099])
def test_sum(ops, n):
    import torch
    a = rand_fr(min(n, 1 << 16), n & 0xffff)
    a = np.tile(a, (-(-n // a.shape[0]), 1))[:n]
    d, want = ops.to_dev(a), orc.fr_sum(a)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        there = [ops.fr_sum(d) for _ in range(3)]
    here = [ops.fr_sum(d) for _ in range(3)]
    torch.cuda.synchronize()
    for t in here + there:
        assert_same(ops.fr_to_host(t)[0], want, "sum")
