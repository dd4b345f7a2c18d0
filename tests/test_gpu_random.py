"""Random elements from a key against a ChaCha20 written here from RFC 8439 (checked by the RFC's own block), and openings that
commit their blinding row through every kind of table."""
import ctypes
import os
import numpy as np
import pytest
import bigref as br
import orc
from gpuutil import rand_fr, assert_same

pytestmark = pytest.mark.gpu

# the host objects are found by their table's address: it stays taken until the process ends
_TABLES = []


@pytest.fixture(scope="module")
def ops():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from grape_amd import ops as o
    o.init(0)
    return o


def _chacha_block(key, counter, nonce):
    def rot(x, n):
        return ((x << n) | (x >> (32 - n))) & 0xffffffff
    init = [0x61707865, 0x3320646e, 0x79622d32, 0x6b206574] + list(key) + [counter] + list(nonce)
    s = list(init)
    for _ in range(10):
        for a, b, c, d in ((0, 4, 8, 12), (1, 5, 9, 13), (2, 6, 10, 14), (3, 7, 11, 15), (0, 5, 10, 15), (1, 6, 11, 12), (2, 7, 8, 13), (3, 4, 9, 14)):
            for x, y, z, n in ((a, b, d, 16), (c, d, b, 12), (a, b, d, 8), (c, d, b, 7)):
                s[x] = (s[x] + s[y]) & 0xffffffff
                s[z] = rot(s[z] ^ s[x], n)
    return [(x + y) & 0xffffffff for x, y in zip(s, init)]


def test_chacha_here_is_the_rfc_s():
    key = np.frombuffer(bytes(range(32)), dtype="<u4").tolist()
    nonce = np.frombuffer(bytes.fromhex("000000090000004a00000000"), dtype="<u4").tolist()
    want = "10f1e7e4d13b5915500fdd1fa32071c4c7d1f4c733c068030422aa9ac3d46c4ed2826446079faa0914c2d705d98b02a2b5129cd1de164eb9cbd083e8a2503c4e"
    assert np.array(_chacha_block(key, 1, nonce), dtype="<u4").tobytes().hex() == want


@pytest.mark.parametrize("n", [1, 64, 65, 500])
def test_random_elements_of_a_key(ops, n):
    import torch
    from grape_amd import _capi
    lib = ops.init()
    words = np.random.default_rng(n).integers(0, 1 << 32, 8, dtype=np.uint64).astype(np.uint32)
    key = (ctypes.c_uint32 * 8)(*[int(x) for x in words])
    out = torch.full((n + 2, 8), -1, dtype=torch.int32, device="cuda")
    _capi.check(lib.grape_fr_random(ops._p(out), n, key, None))
    bits = br.R_MOD.bit_length()
    want, retried = [], 0
    for i in range(n):
        for t in range(128):
            b = _chacha_block(key, t // 2, [i, 0, 0])[8 * (t % 2):8 * (t % 2) + 8]
            x = sum(w << (32 * k) for k, w in enumerate(b)) & ((1 << bits) - 1)
            if x < br.R_MOD:
                break
            retried += 1
        want.append(x)
    assert_same(ops.fr_to_host(out)[:n], np.array(br.ints_to_limbs(want, 4), dtype=np.uint64), "elements")
    assert bool((out[n:] == -1).all()) and (n < 100 or retried > 10)


@pytest.mark.parametrize("n,budget,rows_of", [(512, None, [1, 1, 1, 2, 1, 2]), (512, "0", [1, 1, 2]), (2048, "1", [2, 1, 1])])
def test_openings_of_a_single_row_through_every_table(ops, monkeypatch, n, budget, rows_of):
    """commitment, blinding row and check of one row: through the reference-format table and then through the row's own; through the
    reference-format one alone, without a budget; through the strided table that a commitment of two rows makes of half of a GiB, beside which the
    row's own does not fit (which path is taken when is counted on the host: tables_of_single_rows in native/stream_order.cpp)"""
    from grape_amd import _host as host
    host.load()
    if budget is not None:
        monkeypatch.setitem(os.environ, "GRAPE_TABLE_BUDGET_GIB", budget)
    table = ops.g1_table_gen(ops.g1_make_generators(rand_fr(n, 920)), 256)
    _TABLES.append(table)
    lg = n.bit_length() - 1
    for i, rows in enumerate(rows_of):
        t, point, c = rand_fr(rows * n, 921 + i), rand_fr(lg + rows - 1, 930 + i), rand_fr(1, 940 + i)
        res, ok = host.hyrax_open_verify(ops.to_dev(t), rows * n, n, table, n, point, c, com_scale=1)
        assert ok
        assert_same(res, orc.partial_eval(t, rows * n, point, rows * n, 0, 1)[0], "value %d" % i)
