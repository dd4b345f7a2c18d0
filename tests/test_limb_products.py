"""The field products of the commitment kernels (host build of grape_amd/csrc/fp30.hpp) and of the round kernels (fr26.hpp) on
operands whose limbs are at the bounds that the columns are laid out for, all signs alike and mixed, against Python
integers: balanced limbs of +-(2^29 + 2) and one lazy operand of twice that; limbs of 2^30 times 2^27."""
import ctypes
import os
import random
import subprocess
import numpy as np
import pytest
import bigref as br

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "limb_products_host.cpp")
BN = br.CURVE == "bn254"
LIB = os.path.join(HERE, "native", "liblimb_products_host_bn254.so" if BN else "liblimb_products_host.so")
P = br.P_MOD
W = 30
EDGE = (1 << 29) + 2


@pytest.fixture(scope="module")
def lib():
    deps = [SRC] + [os.path.join(HERE, "..", "grape_amd", "csrc", f) for f in ("fp30.hpp", "fr26.hpp", "divstep.hpp", "curve.hpp", "field.hpp")]
    if not os.path.exists(LIB) or any(os.path.getmtime(d) > os.path.getmtime(LIB) for d in deps):
        subprocess.check_call(["g++", "-O2", "-std=c++17", "-fwrapv", "-fPIC", "-shared", "-Wno-unknown-pragmas"]
                              + (["-DGRAPE_CURVE_BN254"] if BN else []) + ["-o", LIB, SRC])
    return ctypes.CDLL(LIB)


def _value(limbs):
    return sum(int(v) << (W * i) for i, v in enumerate(limbs))


def _operands(n, bound, rng, count):
    """limb vectors: the extremes with all signs alike and alternating, and random ones; a top limb of a few p"""
    top = (4 * P) >> (W * (n - 1))
    out = [np.zeros(n, dtype=np.int32)]
    for sign in (1, -1):
        out.append(np.array([sign * bound] * (n - 1) + [sign * top], dtype=np.int32))
        out.append(np.array([sign * bound * (-1) ** i for i in range(n - 1)] + [sign * top], dtype=np.int32))
    for _ in range(count):
        out.append(np.array([rng.choice([bound, -bound, rng.randint(-bound, bound)]) for _ in range(n - 1)] + [rng.randint(-top, top)], dtype=np.int32))
    return out


def _ptr(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int32))


def _apply(lib, op, a, b, s, u):
    out = np.zeros(lib.fp30_limbs(), dtype=np.int32)
    lib.fp30_apply(op, _ptr(a), _ptr(b), _ptr(s), _ptr(u), _ptr(out))
    return out


def test_products_at_the_bounds_of_their_columns(lib):
    n, rng = lib.fp30_limbs(), random.Random(5)
    rinv = pow(1 << (W * n), -1, P)
    balanced, lazy = _operands(n, EDGE, rng, 12), _operands(n, 2 * EDGE, rng, 6)
    formulas = {0: lambda a, b, s, u: a * b * rinv, 1: lambda a, b, s, u: a * b * rinv, 2: lambda a, b, s, u: a * b * rinv,
                3: lambda a, b, s, u: a * b * rinv - s, 4: lambda a, b, s, u: (a * b - s * u) * rinv, 5: lambda a, b, s, u: a * a * rinv,
                6: lambda a, b, s, u: a * a * rinv, 7: lambda a, b, s, u: a * a * rinv - s - 2 * u}
    for op, want in formulas.items():
        for a in balanced + (lazy if op == 0 else []):
            for b in balanced:
                s, u = (rng.choice(balanced) for _ in range(2)) if rng.random() < 0.7 else (a, b)
                got = _apply(lib, op, a, b, s, u)
                assert (_value(got) - want(*(_value(x) for x in (a, b, s, u)))) % P == 0, op
                # balanced, so that the next product may take it
                assert max(abs(int(v)) for v in got[:-1]) <= EDGE, op
                if op in (0, 2, 6):
                    assert abs(_value(got)) < P, op


def test_carries_and_zero(lib):
    n, rng = lib.fp30_limbs(), random.Random(6)
    zero = np.zeros(n, dtype=np.int32)
    for op, bound in ((8, (3 << 29) - 1), (11, (1 << 31) - 1)):
        for a in _operands(n, bound, rng, 40):
            b = _apply(lib, op, a, zero, zero, zero)
            assert _value(b) == _value(a) and max(abs(int(v)) for v in b[:-1]) <= EDGE
    for a in _operands(n, (1 << 31) - 1, rng, 40):
        m = _apply(lib, 9, a, zero, zero, zero)
        assert _value(m) == _value(a) and all(0 <= int(v) < 1 << W for v in m[:-1])
    rinv = pow(1 << (W * n), -1, P)
    unit = np.array([1] + [0] * (n - 1), dtype=np.int32)
    for k in range(-3, 4):
        # multiples of p are zero as factors, their neighbours are not
        v, limbs = k * P, []
        for _ in range(n - 1):
            d = ((v + (1 << (W - 1))) & ((1 << W) - 1)) - (1 << (W - 1))
            limbs.append(d)
            v = (v - d) >> W
        a = np.array(limbs + [v], dtype=np.int32)
        for f in _operands(n, EDGE, rng, 4):
            assert lib.fp30_zero(_ptr(a), _ptr(f)) == 1
            assert lib.fp30_zero(_ptr(a + unit), _ptr(f)) == int(_value(f) % P == 0)
            c = _apply(lib, 10, a + unit, f, zero, zero)
            assert _value(c) == _value(f) * rinv % P and all(0 <= int(x) < 1 << W for x in c[:-1])


def test_scalar_product_in_wide_digits(lib):
    n, r, w, rng = 10, br.R_MOD, 26, random.Random(7)
    value = lambda limbs: sum(int(v) << (w * i) for i, v in enumerate(limbs))
    top = (2 * r) >> (w * (n - 1))
    # e * x with e below 16 r (limbs below 2^30) and x a difference of two elements or a sum of two (limbs below 2^27)
    es = [np.zeros(n, dtype=np.int32), np.array([(1 << 30) - 16] * (n - 1) + [8 * top], dtype=np.int32)]
    es += [np.array([rng.randrange(1 << 30) for _ in range(n - 1)] + [rng.randrange(8 * top)], dtype=np.int32) for _ in range(10)]
    bound = (1 << 27) - 1
    xs = [np.array([s * bound] * (n - 1) + [s * top], dtype=np.int32) for s in (1, -1)] + [np.zeros(n, dtype=np.int32)]
    xs += [np.array([rng.randint(-bound, bound) for _ in range(n - 1)] + [rng.randint(-top, top)], dtype=np.int32) for _ in range(20)]
    out = np.zeros(n, dtype=np.int32)
    for e in es:
        for x in xs:
            for add_r in (0, 1, 4, 31):
                lib.fr26_product(_ptr(e), _ptr(x), add_r, _ptr(out))
                v, exact = value(out), value(e) * value(x)
                assert (v * (1 << (w * n)) - exact) % r == 0
                assert all(0 <= int(d) < 1 << w for d in out[:-1])
                # between exact / 2^260 + add_r r and (1 + 2^-20) r above
                low = v * (1 << (w * n)) - exact - add_r * r * (1 << (w * n))
                assert 0 <= low < r * ((1 << (w * n)) + (1 << (w * n - 20)))


def test_limb_sums_at_their_bounds(lib):
    """sums of up to 31 elements and of 16 differences, with the largest limbs that elements have: 24 are what a thread of the carried
    rounds adds up"""
    n, r, w, rng = 10, br.R_MOD, 26, random.Random(8)
    limbs = lambda v: np.array([(v >> (w * i)) & ((1 << w) - 1) for i in range(n)], dtype=np.int32)
    ones = (1 << (w * (n - 1))) - 1                      # the low limbs all ones
    elements = [0, 1, r - 1, ones, (((r >> (w * (n - 1))) - 1) << (w * (n - 1))) + ones, rng.randrange(r)]
    out = np.zeros(8, dtype=np.uint32)

    def check(total, add_r, want):
        assert np.abs(total + add_r * limbs(r).astype(np.int64)).max() < 1 << 31
        lib.fr26_limb_sum(_ptr(total.astype(np.int32)), add_r, out.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)))
        assert sum(int(x) << (32 * i) for i, x in enumerate(out)) == want % r

    for count in (1, 16, 24, 31):
        for v in elements:
            check(count * limbs(v).astype(np.int64), 0, count * v)
        mixed = [rng.choice(elements + [rng.randrange(r)]) for _ in range(count)]
        check(sum(limbs(v).astype(np.int64) for v in mixed), 0, sum(mixed))
    for a in elements:
        for b in elements:
            check(16 * (limbs(a).astype(np.int64) - limbs(b)), 16, 16 * (a - b))
