"""Short copies to the host around the size that goes through pinned memory, and the handing-on of default-stream blocks:
in stream order while only known streams are about, with a wait otherwise."""
import ctypes
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    from grape_amd import _capi, ops
    ops.init(0)
    return _capi.load()


@pytest.mark.parametrize("nbytes", [1, 4, 6, 32, 1020, 1024, 16384, 16388, 40000])
@pytest.mark.parametrize("offset", [0, 4, 2])
def test_short_copies(lib, nbytes, offset):
    src = torch.randint(0, 256, (nbytes + 8,), dtype=torch.uint8, device="cuda")
    out = np.zeros(nbytes, dtype=np.uint8)
    assert lib.grape_memcpy_d2h(out.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(src.data_ptr() + offset), nbytes, None) == 0
    assert np.array_equal(out, src.cpu().numpy()[offset:offset + nbytes])


@pytest.mark.parametrize("pinned", [False, True])
def test_short_copies_of_host_memory(lib, pinned):
    """a source that is host memory stays with the runtime's copy, which serves pinned memory and refuses the rest: no kernel reads it"""
    src = torch.arange(64, dtype=torch.int32)
    src = src.pin_memory() if pinned else src
    out = np.zeros(64, dtype=np.int32)
    rc = lib.grape_memcpy_d2h(out.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(src.data_ptr()), 256, None)
    assert rc == (0 if pinned else -2)
    assert np.array_equal(out, src.numpy() if pinned else np.zeros(64, dtype=np.int32))
    dev = torch.arange(64, dtype=torch.int32, device="cuda")
    assert lib.grape_memcpy_d2h(out.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(dev.data_ptr()), 256, None) == 0
    assert np.array_equal(out, np.arange(64))


def test_short_copy_of_the_last_bytes_of_a_block(lib):
    from grape_amd import _capi
    p = ctypes.c_void_p()
    _capi.check(lib.grape_malloc(ctypes.byref(p), 1 << 21))
    block = np.random.default_rng(5).integers(0, 1 << 31, 1 << 19).astype(np.int32)
    _capi.check(lib.grape_memcpy_h2d(p, block.ctypes.data_as(ctypes.c_void_p), 1 << 21, None))
    out = np.zeros(64, dtype=np.int32)
    dst = out.ctypes.data_as(ctypes.c_void_p)
    assert lib.grape_memcpy_d2h(dst, ctypes.c_void_p(p.value + (1 << 21) - 256), 256, None) == 0
    assert np.array_equal(out, block[-64:])
    _capi.check(lib.grape_free(p))


def _cycle(lib, n_words, value):
    """fill a block, queue its copy into a second one, give the first back and take it again for other contents"""
    from grape_amd import _capi
    p, q = ctypes.c_void_p(), ctypes.c_void_p()
    host = np.full(n_words, value, dtype=np.uint32)
    _capi.check(lib.grape_malloc_on_default(ctypes.byref(p), 4 * n_words))
    _capi.check(lib.grape_malloc_on_default(ctypes.byref(q), 4 * n_words))
    _capi.check(lib.grape_memcpy_h2d(p, host.ctypes.data_as(ctypes.c_void_p), 4 * n_words, None))
    _capi.check(lib.grape_memcpy_d2d(q, p, 4 * n_words, None))
    _capi.check(lib.grape_free_on_default(p))
    r = ctypes.c_void_p()
    _capi.check(lib.grape_malloc_on_default(ctypes.byref(r), 4 * n_words))
    _capi.check(lib.grape_memset_zero(r, 4 * n_words, None))
    got = np.zeros(n_words, dtype=np.uint32)
    _capi.check(lib.grape_memcpy_d2h(got.ctypes.data_as(ctypes.c_void_p), q, 4 * n_words, None))
    again = r.value == p.value
    for b in (q, r):
        _capi.check(lib.grape_free_on_default(b))
    assert np.array_equal(got, host)
    return again


@pytest.mark.parametrize("n_words", [1, 1000, 1 << 22])
def test_default_blocks_are_handed_on(lib, n_words):
    for k in range(4):
        assert _cycle(lib, n_words, 7 + k)
    from grape_amd import ops
    h = ops.stream_create()                       # a stream the library cannot vouch for: the same contents, with waits
    try:
        for k in range(4):
            _cycle(lib, n_words, 70 + k)
    finally:
        ops.stream_destroy(h)
    p = ctypes.c_void_p()                         # a block of the other kind is taken over as well
    assert lib.grape_malloc(ctypes.byref(p), 4 * n_words) == 0 and lib.grape_free(p) == 0
    _cycle(lib, n_words, 700)


def _late_reader(lib, reader, take, writer):
    """Copies of a 256 MB block are queued on `reader`, the block is given back as a default-stream block, taken again with `take`
    and overwritten on `writer`: the copies hold the old contents."""
    from grape_amd import _capi
    words = 1 << 26
    p, q = ctypes.c_void_p(), ctypes.c_void_p()
    _capi.check(lib.grape_malloc_on_default(ctypes.byref(p), 4 * words))
    _capi.check(lib.grape_malloc(ctypes.byref(q), 4 * words))
    host = np.arange(words, dtype=np.uint32)
    _capi.check(lib.grape_memcpy_h2d(p, host.ctypes.data_as(ctypes.c_void_p), 4 * words, None))
    _capi.check(lib.grape_memset_zero(q, 4 * words, None))
    _capi.check(lib.grape_stream_sync(None))
    for _ in range(8):
        _capi.check(lib.grape_memcpy_d2d(q, p, 4 * words, reader))
    _capi.check(lib.grape_free_on_default(p))
    r = ctypes.c_void_p()
    _capi.check(take(ctypes.byref(r), 4 * words))
    assert r.value == p.value
    _capi.check(lib.grape_memset_zero(r, 4 * words, writer))
    for s in (reader, writer):
        _capi.check(lib.grape_stream_sync(s))
    got = np.empty(words, dtype=np.uint32)
    _capi.check(lib.grape_memcpy_d2h(got.ctypes.data_as(ctypes.c_void_p), q, 4 * words, None))
    for b in (q, r):
        _capi.check(lib.grape_free(b))
    assert np.array_equal(got, host)


def test_a_block_is_not_overwritten_under_a_reader(lib):
    from grape_amd import ops
    user = ops.stream_create()                    # reads a block that the default stream takes over
    try:
        _late_reader(lib, user, lib.grape_malloc_on_default, None)
    finally:
        ops.stream_destroy(user)
    side = ops.stream_create()                    # joined by this test itself: a block the default stream reads goes to another stream
    try:
        assert lib.grape_stream_internal(side) == 0
        _late_reader(lib, None, lib.grape_malloc, side)
        _late_reader(lib, None, lib.grape_malloc_on_default, None)
    finally:
        ops.stream_destroy(side)
