"""Two carried rounds in one pass against the same two rounds one after the other, bit for bit: periods that fill no wave, a single
period, several workgroups and steps, every kind of first round, and the elements and challenges with the largest limbs."""
import ctypes
import numpy as np
import pytest
import bigref as br
from gpuutil import rand_fr, assert_same

pytestmark = pytest.mark.gpu


class Carried(ctypes.Structure):
    _fields_ = [("A_out", ctypes.c_void_p), ("Z_out", ctypes.c_void_p), ("A", ctypes.c_void_p), ("Z", ctypes.c_void_p),
                ("idx1", ctypes.c_void_p), ("halves", ctypes.c_void_p), ("len", ctypes.c_uint32), ("eq", ctypes.c_void_p),
                ("eq_high", ctypes.c_void_p), ("period", ctypes.c_uint32), ("n_out", ctypes.c_uint32), ("tab_a", ctypes.c_void_p),
                ("tab_z", ctypes.c_void_p), ("plain_sums", ctypes.c_int), ("partial", ctypes.c_void_p), ("pair", ctypes.c_uint32)]


@pytest.fixture(scope="module")
def ops():
    from grape_amd import ops
    ops.init(0)
    return ops


def _elements(n, seed, largest):
    x = rand_fr(n, seed)
    if largest:                                              # r - 1 in memory, and zero
        x[:] = np.frombuffer((br.R_MOD - 1).to_bytes(32, "little"), dtype=np.uint64)
        x[seed % 3::5] = 0
    return x


@pytest.mark.parametrize("kind", ["gather", "enter", "later", "later_plain"])
@pytest.mark.parametrize("period,periods,largest", [(1, 1, False), (31, 3, False), (33, 1, True), (257, 40, False), (4096, 25, True), (11008, 128, False),
                                                    (1 << 16, 2, False), (1 << 16, 75, True)])
def test_pair_is_two_rounds(ops, kind, period, periods, largest):
    import torch
    from grape_amd import _capi
    lib = ops.init()
    n, length = period * periods, 100                        # elements left, table entries
    A, Z = ops.to_dev(_elements(4 * n, 1, largest)), ops.to_dev(_elements(4 * n, 2, largest))
    eq, high = ops.to_dev(_elements(period, 3, largest)), ops.to_dev(_elements(2 * periods, 4, largest))
    halves = ops.to_dev(_elements(4 * length, 5, largest))
    idx = torch.randint(0, length + 1, (4 * n,), device="cuda", dtype=torch.int32, generator=torch.Generator("cuda").manual_seed(6))
    ch = ops.to_dev(_elements(4, 7, largest))
    tabs = torch.empty(4 * 100, dtype=torch.int32, device="cuda")
    _capi.check(lib.grape_fold_tables(tabs.data_ptr(), ch.data_ptr(), 4, None))

    def proof(pair):
        a_out, z_out = A.clone(), Z.clone()                  # in place, as the proofs run them
        r = (Carried * 2)()
        for i in range(2):
            r[i] = Carried(a_out.data_ptr(), z_out.data_ptr(), a_out.data_ptr(), z_out.data_ptr(), None, None, 0, eq.data_ptr(), None, period,
                           2 * n >> i, tabs.data_ptr() + 800 * i, tabs.data_ptr() + 800 * i + 400, 0 if kind in ("enter", "later") else 1, None,
                           (i + 1) if pair else 0)
        if kind == "gather":
            r[0].idx1, r[0].halves, r[0].len = idx.data_ptr(), halves.data_ptr(), length
        if kind in ("gather", "enter"):
            r[0].eq_high = high.data_ptr()
        sums = torch.zeros((10, 8), dtype=torch.int32, device="cuda")
        parts = [torch.empty(lib.grape_carried_partial_bytes(ctypes.byref(x)) // 4, dtype=torch.int32, device="cuda") for x in r]
        for x, p in zip(r, parts):
            x.partial = p.data_ptr()
        if pair:
            _capi.check(lib.grape_carried_queue_pair(ctypes.byref(r[0]), ctypes.byref(r[1]), None))
        else:
            for x in r:
                _capi.check(lib.grape_carried_queue(ctypes.byref(x), None))
        for i, x in enumerate(r):
            _capi.check(lib.grape_carried_finish(sums.data_ptr() + 160 * i, 5, ctypes.byref(x), 1, None))
        torch.cuda.synchronize()
        return ops.fr_to_host(sums), ops.fr_to_host(a_out)[:n], ops.fr_to_host(z_out)[:n]

    for g, w, what in zip(proof(True), proof(False), ("sums", "A", "Z")):
        assert_same(g, w, what)


def test_wrong_pairs_are_refused(ops):
    lib = ops.init()
    r = (Carried * 2)()
    for i in range(2):
        r[i].period, r[i].n_out, r[i].pair = 4, 16 >> i, i + 1
    assert lib.grape_carried_queue_pair(ctypes.byref(r[1]), ctypes.byref(r[0]), None) != 0      # the other way round
    assert lib.grape_carried_queue(ctypes.byref(r[0]), None) != 0                                # half a pass
    r[1].n_out = 16
    assert lib.grape_carried_queue_pair(ctypes.byref(r[0]), ctypes.byref(r[1]), None) != 0      # no fold of the first
