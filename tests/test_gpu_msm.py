"""Window sums of a sum of scalar multiples of arbitrary points (grape_g1_msm_windows), combined here in Python integers,
against the oracle's row commitment over the same points."""
import numpy as np
import pytest
import bigref as br

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _combine(windows):
    w = windows.cpu().numpy().view(np.uint64).reshape(64, 4, -1)
    acc = None
    for s in w[::-1]:
        for _ in range(4):
            acc = br.g1_add(acc, acc)
        x, y, zz, zzz = (br.fp_unpack(c.reshape(1, -1))[0] for c in s)
        if zz:
            acc = br.g1_add(acc, (x * pow(zz, -1, br.P_MOD) % br.P_MOD, y * pow(zzz, -1, br.P_MOD) % br.P_MOD))
    return acc


@pytest.fixture(scope="module")
def setup():
    import orc
    from gpuutil import rand_fr
    from grape_amd import ops
    ops.init(0)
    gens = orc.g1_make_generators(rand_fr(130, 601))
    return ops, orc, rand_fr, gens


@pytest.mark.parametrize("n", [1, 2, 16, 63, 64, 65, 130])
def test_against_the_oracle(setup, n):
    ops, orc, rand_fr, gens = setup
    k = rand_fr(n, 602 + n)
    small = br.fr_pack([0, 1, br.R_MOD - 1, (br.R_MOD - 1) // 2, (br.R_MOD + 1) // 2, 8, br.R_MOD - 8])
    k[: min(n, 7)] = small[: min(n, 7)] if n > 2 else k[: min(n, 7)]
    pts = gens[:n].copy()
    if n >= 63:
        pts[20] = 0                                          # the identity among the points
        pts[31] = pts[30]                                    # the same point and scalar twice, and its negative
        k[31] = k[30]
        k[33] = br.fr_pack([br.R_MOD - br.fr_unpack(k[30:31])[0]])[0]
        pts[33] = pts[30]
    jac = ops.g1_affine_to_jacobian(ops.to_dev(pts))
    got = _combine(ops.g1_msm_windows(jac, ops.to_dev(k)))
    want = orc.commit_fr(k, orc.g1_table(pts, 256), n, n)
    assert got == br.g1_unpack(want)[0]


def test_more_points_than_one_slab(setup):
    """32 768 + 65 points: the same 64 points over and over, so the oracle's sum has 64 terms"""
    ops, orc, rand_fr, gens = setup
    n = 32768 + 65
    k = rand_fr(n, 699)
    idx = np.arange(n) % 64
    jac = ops.g1_affine_to_jacobian(ops.to_dev(np.ascontiguousarray(gens[idx])))
    got = _combine(ops.g1_msm_windows(jac, ops.to_dev(k)))
    vals = br.fr_unpack(k)
    sums = [0] * 64
    for i, v in zip(idx, vals):
        sums[i] = (sums[i] + v) % br.R_MOD
    want = orc.commit_fr(br.fr_pack(sums), orc.g1_table(gens[:64], 256), 64, 64)
    assert got == br.g1_unpack(want)[0]
