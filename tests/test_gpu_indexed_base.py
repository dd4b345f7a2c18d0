"""Rows committed through their table indices with a base entry that costs nothing, against the oracle's commitment of the values:
rows of the base entry alone, without it, elements outside the table, one and several column segments, both orders of the rows."""
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


@pytest.fixture(scope="module")
def tables(ops):
    gens = ops.g1_make_generators(rand_fr(256, 801))
    return gens, ops.g1_wide_table_gen(gens, 8, 32, 128), orc.g1_table(ops.g1_to_host(gens), 256)


@pytest.mark.parametrize("length,base", [(1, 0), (2, 0), (2, 1), (8, 3), (64, 63)])
def test_tables_of_a_power_of_two(ops, tables, length, base):
    """the last index is the digit 2^(c-1) of its radix 2^c: it stays positive"""
    test_base_entry(ops, tables, 7, 65, 0, length, base)


@pytest.mark.parametrize("rows,cols,uneven", [(1, 1, 0), (1, 256, 1), (5, 65, 0), (37, 256, 1), (64, 100, 0), (600, 64, 1), (600, 128, 0)])
def test_base_entry(ops, tables, rows, cols, uneven, length=9, base=3):
    import torch
    from grape_amd import _capi
    lib = ops.init()
    gens, wide, ref = tables
    B = rand_fr(length, 802)
    rng = np.random.default_rng(rows * cols)
    idx = rng.integers(0, length + 1, (rows, cols)).astype(np.int32)      # 0 is outside the table
    idx[0::4] = base + 1
    idx[1::4, cols // 2:] = base + 1
    idx[2::4][idx[2::4] == base + 1] = 0
    less = orc.vec2("orc_fr_vec_sub", B, np.repeat(B[base:base + 1], length, axis=0))
    scaled = torch.empty(lib.grape_g1_wide_table_bytes(cols, 1, length) // 4, dtype=torch.int32, device="cuda")
    d_less = ops.to_dev(less)
    _capi.check(lib.grape_g1_scaled_table_gen(scaled.data_ptr(), d_less.data_ptr(), length, cols, wide.data_ptr(), 256, 8, 32, 128, None))
    # every row starts at sum_i B_base G_i; elements outside the table then stand for B_base too
    point = ops.to_dev(orc.commit_fr(np.repeat(B[base:base + 1], cols, axis=0), ref, cols, 256))
    start = torch.empty(64, dtype=torch.int32, device="cuda")
    _capi.check(lib.grape_commit_start(start.data_ptr(), point.data_ptr(), None))
    d_idx, out = torch.from_numpy(idx).cuda(), ops.g1_empty(rows)
    flag = torch.zeros(1, dtype=torch.int32, device="cuda")
    _capi.check(lib.grape_commit_indexed(out.data_ptr(), d_idx.data_ptr(), rows * cols, cols, scaled.data_ptr(), cols, length, base + 1,
                                         start.data_ptr(), uneven, flag.data_ptr(), None))
    torch.cuda.synchronize()
    values = B[np.where(idx == 0, base, idx - 1).ravel()]
    assert int(flag) == 0
    assert_same(ops.g1_to_host(out), orc.commit_fr(values, ref, cols, 256), "commitments")


# the host objects are found by their table's address: it stays taken until the process ends
_TABLES = []


@pytest.mark.parametrize("first", ["padded", "even"])
def test_ranges_whose_rows_are_the_lowest_key(ops, first):
    """one lookup object for witnesses that it pads and others, in both orders: its table is made for the first of them.  beta is the
    table's size, so B[low] = 2 B[0]: a row of nothing but the lowest key adds its start to a sum that is equal to it"""
    import torch
    from grape_amd import _host as host
    host.load()
    N, low, msm = 16, -8, 64
    table = ops.g1_table_gen(ops.g1_make_generators(rand_fr(msm, 830 if first == "padded" else 831)), 256)
    _TABLES.append(table)
    rng = np.random.default_rng(832)
    host.set_input_format("i32")
    try:
        for turn, kind in enumerate([first, "even" if first == "padded" else "padded", first]):
            D, lg = (2 * 11008, 15) if kind == "padded" else (1 << 14, 14)
            x = rng.integers(low, -low, D).astype(np.int32)
            x[:4 * msm] = low
            x[5 * msm:6 * msm] = 0
            x[7 * msm:8 * msm] = -low - 1
            args = (torch.from_numpy(x).cuda(), D, low, N, rand_fr(1, 833 + turn), rand_fr(lg, 840 + turn), rand_fr(lg, 850 + turn), table, msm, 1, msm)
            got = host.tlookup_range_prove(*args, want_commitments=True)
            host.set_indexed_commit(False)
            want = host.tlookup_range_prove(*args, want_commitments=True)
            host.set_indexed_commit(True)
            for k in ("transcript", "S_claim", "com_A", "com_m"):
                assert_same(got[k], want[k], "%s, %s" % (kind, k))
    finally:
        host.set_indexed_commit(True)
        host.set_input_format("fr")
