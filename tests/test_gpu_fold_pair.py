"""Two folds side by side and the short passes (16 or 256 threads an output) against the oracle: ragged axes, one and several
outer indices, in place, from a kept tensor and from integers, passes of the same and of different kinds."""
import ctypes
import numpy as np
import pytest
import orc
from gpuutil import rand_fr, assert_same

pytestmark = pytest.mark.gpu


class FoldJob(ctypes.Structure):
    _fields_ = [("t", ctypes.c_void_p), ("from_", ctypes.c_void_p), ("ints", ctypes.c_void_p), ("N", ctypes.c_size_t),
                ("x", ctypes.c_void_p), ("c", ctypes.c_uint32), ("id", ctypes.c_uint32), ("gap", ctypes.c_uint32)]


@pytest.fixture(scope="module")
def ops():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from grape_amd import ops as o
    o.init(0)
    return o


# (source, outer, c, gap, first challenge)
SHAPES = {
    "one_thread_an_output": ("t", 1, 3, 70000, 1),
    "slab": ("t", 3, 15, 16, 0),
    "two_variables": ("from", 5, 4, 500, 2),
    "nothing_to_bind": ("from", 7, 1, 9, 0),
    "ragged_16": ("t", 1, 200, 17, 3),
    "ragged_16_rows": ("from", 32, 129, 128, 1),
    "eval": ("t", 1, 4096, 1, 0),
    "eval_ragged": ("from", 1, 4095, 1, 0),
    "rows_256": ("t", 33, 257, 1, 2),
    "ints_16": ("ints", 32, 100, 33, 1),
    "ints_256": ("ints", 1, 6000, 1, 0),
    "ints_rows": ("ints", 2, 300, 250, 0),
    "nine_variables": ("t", 1, 512, 3, 0),
    "seventeen_variables": ("from", 1, 70001, 1, 0),
    # one workgroup's steps of 256 outputs: eight and nine, one slab and several, field elements and integers
    "steps_9_of_512": ("t", 1, 512, 1, 0),
    "steps_9_of_300": ("from", 1, 300, 1, 1),
    "steps_10_of_513": ("t", 1, 513, 1, 0),
    "steps_9_of_several": ("from", 3, 300, 1, 0),
    "steps_8": ("t", 1, 128, 8, 2),
    "steps_8_of_several": ("from", 17, 100, 8, 0),
    "steps_7": ("t", 256, 64, 16, 0),
    "steps_9_of_2048": ("from", 1, 32, 64, 0),
    "steps_5_ragged": ("t", 2, 17, 30, 1),
    "steps_7_of_ints": ("ints", 5, 64, 16, 0),
}


@pytest.mark.parametrize("pair", [("one_thread_an_output", "slab"), ("two_variables", "nothing_to_bind"), ("ragged_16", "ragged_16_rows"),
                                  ("eval", "eval_ragged"), ("rows_256", "eval"), ("ints_16", "ints_256"), ("ints_rows", "ragged_16"),
                                  ("nine_variables", "seventeen_variables"), ("nothing_to_bind", "ints_rows"), ("seventeen_variables",),
                                  ("ints_256",), ("steps_9_of_512",), ("steps_9_of_300",), ("steps_10_of_513",), ("steps_9_of_several",), ("steps_8",),
                                  ("steps_8_of_several",), ("steps_7",), ("steps_9_of_2048",), ("steps_5_ragged",), ("steps_7_of_ints",),
                                  ("steps_9_of_512", "steps_8_of_several")], ids="-".join)
def test_folds_side_by_side(ops, pair):
    import torch
    from grape_amd import _capi
    lib = ops.init()
    jobs = (FoldJob * len(pair))()
    keep, want, out = [], [], []
    for k, name in enumerate(pair):
        src, outer, c, gap, idx = SHAPES[name]
        n = outer * c * gap
        x = rand_fr(idx + 18, 40 + k)
        if src == "ints":
            ints = np.random.default_rng(50 + k).integers(-(1 << 31), 1 << 31, n, dtype=np.int64).astype(np.int32)
            ints[:3] = [-(1 << 31), (1 << 31) - 1, 0]
            d, host = torch.from_numpy(ints).cuda(), orc.from_i32(ints)
        else:
            host = rand_fr(n, 60 + k)
            d = ops.to_dev(host)
        t = d if src == "t" else torch.full((max(1, lib.grape_fr_fold_i32_elems(n, c, gap)), 8), -1, dtype=torch.int32, device="cuda")
        dx = ops.to_dev(x)
        jobs[k] = FoldJob(t.data_ptr(), d.data_ptr() if src == "from" else None, d.data_ptr() if src == "ints" else None, n, dx.data_ptr(), c, idx, gap)
        keep.append((d, d.clone(), dx, src))
        out.append((t, outer * gap))
        want.append(orc.partial_eval(host, n, x, c, idx, gap)[:outer * gap])
    _capi.check(lib.grape_fr_fold_pair(jobs, len(pair), None))
    torch.cuda.synchronize()
    for (t, n), w, name, (d, before, _, src) in zip(out, want, pair, keep):
        assert_same(ops.fr_to_host(t)[:n], w, name)
        assert src == "t" or torch.equal(d, before)


def test_bad_pairs_are_refused(ops):
    lib = ops.init()
    assert lib.grape_fr_fold_pair(None, 1, None) != 0
    jobs = (FoldJob * 3)()
    assert lib.grape_fr_fold_pair(jobs, 0, None) != 0 and lib.grape_fr_fold_pair(jobs, 3, None) != 0
