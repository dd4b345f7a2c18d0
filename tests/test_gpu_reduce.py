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
