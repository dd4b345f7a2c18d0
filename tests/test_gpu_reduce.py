"""Row reduction of a commitment at the edges of its plan: one row and many, one partial sum and many groups, rows that
share no workgroup, and partial sums that are equal, opposite or the identity (the exceptional additions)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup():
    import orc
    from gpuutil import rand_fr
    from grape_amd import ops
    ops.init(0)
    gens = ops.g1_make_generators(rand_fr(128, 501))
    table = ops.g1_wide_table_gen(gens, 8, 2, 128)
    ref = orc.g1_table(orc.g1_make_generators(rand_fr(128, 501)), 256)
    return ops, orc, table, ref


# rows x columns: around the lines of geom::reduce_plan (512, 1024, 2048, 4096, 8192 rows) and of wide_plan's segments
@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 128), (3, 128), (511, 128), (513, 100), (1025, 65), (2049, 7), (4097, 5), (8192, 3), (8193, 3)])
def test_rows_of_every_plan(setup, rows, cols):
    ops, orc, table, ref = setup
    w = np.random.default_rng(rows).integers(-(1 << 14), 1 << 14, (rows, cols)).astype(np.int32)
    w[rows // 2] = 0                                        # a row that commits to the identity
    got = ops.g1_to_host(ops.commit_i32(torch.from_numpy(w).cuda(), cols, table, 128, 8, 2, 128))
    some = sorted({0, rows // 2, rows - 1, rows // 3, 2 * rows // 3})
    assert np.array_equal(got[some], orc.commit_i32(np.ascontiguousarray(w[some]), ref, cols, 128))


def test_equal_and_opposite_partial_sums(setup):
    """all generators the same point: every lane holds +-w * G, so the tree meets doublings and cancellations"""
    ops, orc, _, _ = setup
    from gpuutil import rand_fr
    k = np.repeat(rand_fr(1, 502), 128, axis=0)
    table = ops.g1_wide_table_gen(ops.g1_make_generators(k), 8, 2, 128)
    ref = orc.g1_table(orc.g1_make_generators(k), 256)
    w = np.zeros((6, 128), dtype=np.int32)
    w[0] = 7                                                # all equal
    w[1] = np.where(np.arange(128) % 2 == 0, 9, -9)         # pairs cancel
    w[2, :64], w[2, 64:] = 5, -5                            # halves cancel inside a lane
    w[3, 0], w[3, 127] = 3, -3
    w[4, ::3] = -11
    for rows in (w, np.tile(w, (1400, 1))):                 # few rows (quads only) and more than 8192 (lanes first)
        got = ops.g1_to_host(ops.commit_i32(torch.from_numpy(rows).cuda(), 128, table, 128, 8, 2, 128))
        want = orc.commit_i32(w, ref, 128, 128)
        assert np.array_equal(got[:6], want) and np.array_equal(got[-6:], want)


@pytest.mark.parametrize("rowlen,rows,live", [(64, 1, 1.0), (100, 33, 0.5), (128, 35, 1.0), (65, 40, 0.02), (128, 3000, 0.7)])
@pytest.mark.parametrize("c,J", [(8, 32), (13, 5), (11, 1)])
def test_masked_strided_commitment(setup, rowlen, rows, live, c, J):
    """flagged-in elements only, through the strided table: the dense commitment of the tensor with the others zeroed (row
    counts around a multiple of 32, full batches, a last partial one, rows with none)"""
    ops, orc, _, _ = setup
    from gpuutil import rand_fr
    gens = ops.g1_make_generators(rand_fr(128, 501))
    nw = (255 + c - 1) // c
    nsets = (nw + J - 1) // J
    table = ops.g1_strided_table_gen(gens, c, J, nsets)
    s = rand_fr(rows * rowlen, 503)
    rng = np.random.default_rng(rows)
    skip = (rng.random(rows * rowlen) >= live).astype(np.int32) * 3
    if rows > 1:
        skip[rowlen: 2 * rowlen] = 1
    got = ops.g1_to_host(ops.commit_fr_strided_masked(ops.to_dev(s), torch.from_numpy(skip).cuda(), rowlen, table, 128, c, J, nsets))
    s[skip != 0] = 0
    want = ops.g1_to_host(ops.commit_fr_strided(ops.to_dev(s), rowlen, table, 128, c, J, nsets))
    assert np.array_equal(got, want)
    assert rows == 1 or not got[1].any()
    ref = orc.g1_table(orc.g1_make_generators(rand_fr(128, 501)), 256)
    assert np.array_equal(got[-1:], orc.commit_fr(s[-rowlen:], ref, rowlen, 128))


# few rows of full-width scalars: the windows go over several waves (window_split: 1, 2, 3, 16 shares, shares of unequal
# length), the partial sums over one, two and three levels of groups
@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 128), (3, 100), (15, 128), (129, 64), (300, 65)])
def test_windows_over_several_waves(setup, rows, cols):
    ops, orc, _, ref = setup
    from gpuutil import rand_fr
    gens = ops.g1_make_generators(rand_fr(128, 501))
    s = rand_fr(rows * cols, 600 + rows)
    s[:: 7] = 0
    some = sorted({0, rows // 2, rows - 1})
    want = orc.commit_fr(np.ascontiguousarray(s.reshape(rows, cols, 4)[some].reshape(-1, 4)), ref, cols, 128)
    d = ops.to_dev(s)
    for c, nw in ((8, 32), (13, 20)):
        got = ops.g1_to_host(ops.commit_fr(d, cols, ops.g1_wide_table_gen(gens, c, nw, 1 << (c - 1)), 128, c, nw, 1 << (c - 1)))
        assert np.array_equal(got[some], want), (c, nw)
    for c, J, nsets in ((11, 1, 24), (8, 5, 7), (8, 32, 1)):
        got = ops.g1_to_host(ops.commit_fr_strided(d, cols, ops.g1_strided_table_gen(gens, c, J, nsets), 128, c, J, nsets))
        assert np.array_equal(got[some], want), (c, J)


def test_one_long_row_in_three_levels(setup):
    """a row of 4096: 64 segments x 10 shares x 64 lanes = 40960 partial sums -> 640 -> 40 -> 1"""
    ops, orc, _, _ = setup
    from gpuutil import rand_fr
    gens = ops.g1_make_generators(rand_fr(4096, 503))
    s = ops.to_dev(rand_fr(4096, 504))
    a = ops.g1_to_host(ops.commit_fr(s, 4096, ops.g1_wide_table_gen(gens, 8, 32, 128), 4096, 8, 32, 128))
    b = ops.g1_to_host(ops.commit_fr_strided(s, 4096, ops.g1_strided_table_gen(gens, 8, 8, 4), 4096, 8, 8, 4))
    c = ops.g1_to_host(ops.commit_fr_ref_table(s, 4096, ops.g1_table_gen(gens, 256), 4096))
    halves = [ops.g1_to_host(ops.commit_fr(s[:2048].contiguous(), 2048, ops.g1_wide_table_gen(gens[:2048].contiguous(), 8, 32, 128), 2048, 8, 32, 128))]
    assert np.array_equal(a, b) and np.array_equal(a, c) and not np.array_equal(a, halves[0])
