"""Every entry of the eq tables of all prefixes, at the sizes where an entry's factors change their place (5 low bits, 11 bits a
workgroup, workgroups of several levels), an entry a thread below those and level by level above them, and the challenge tables' rows: both against their definitions."""
import numpy as np
import pytest
import bigref as br
import orc
from gpuutil import rand_fr, assert_same

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from grape_amd import ops
    ops.init(0)
    return ops


@pytest.mark.parametrize("nu", [0, 1, 2, 3, 4, 5, 6, 7, 10, 11, 12, 13, 14, 18, 19, 20, 21])
def test_every_level(ops, nu):
    u = rand_fr(max(nu, 1), 300 + nu)[:nu]
    if nu > 3:
        u[1], u[nu - 1] = br.fr_pack([0])[0], br.fr_pack([1])[0]      # factors 0 and 1
    level, levels = br.fr_pack([1]), []
    for j in range(nu + 1):
        levels.append(level)
        if j < nu:
            hi = orc.vec2("orc_fr_vec_mul", level, np.repeat(u[j:j + 1], len(level), axis=0))
            lo = orc.vec2("orc_fr_vec_sub", level, hi)
            level = np.concatenate([lo, hi])
    got = ops.fr_to_host(ops.eq_pyramid(ops.to_dev(u) if nu else ops.to_dev(rand_fr(1, 1)), nu))
    assert_same(got, np.concatenate(levels), "pyramid")


@pytest.mark.parametrize("count", [1, 7, 64])
def test_challenge_tables(ops, count):
    import torch
    from grape_amd import _capi
    v = rand_fr(count, 310)
    v[0] = br.fr_pack([br.R_MOD - 1])[0]
    tabs = torch.empty(100 * count, dtype=torch.int32, device="cuda")
    _capi.check(ops.init().grape_fold_tables(tabs.data_ptr(), ops.to_dev(v).data_ptr(), count, None))
    got = tabs.cpu().numpy().reshape(count, 10, 10)
    for k, x in enumerate(br.fr_unpack(v)):
        for j in range(10):
            w = x * (1 << (26 * j + 52)) % br.R_MOD
            assert [int(t) for t in got[k, j]] == [(w >> (26 * i)) & ((1 << 26) - 1) for i in range(10)], (k, j)
