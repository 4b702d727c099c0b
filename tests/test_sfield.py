"""Signed field arithmetic of the ladders (csrc/sfield.hpp), host build, against Python integers:
random limbs and limbs at the ends of their ranges, for the three field primes."""
import ctypes
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "wgpu-sigops_amd", "csrc")
P = [2**256 - 2**32 - 977, 2**256 - 2**224 + 2**192 + 2**96 - 1, 2**255 - 19]
N = 2**29 - 1
RINV = [pow(2**261, -1, p) for p in P]


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("sfield") / "libsfield.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-DSIGOPS_HOST_CHECK=1",
                    "-I" + CSRC, "-o", so, os.path.join(HERE, "devcheck", "sfield_check.cpp")], check=True)
    return ctypes.CDLL(so)


def value(limbs):
    return sum(x << (29 * k) for k, x in enumerate(limbs))


def vectors(rng, lo, hi, count):
    """limb vectors: all lowest, all highest, alternating, zero, one, then random; top limb small"""
    top = 1 << 26
    fixed = [[lo] * 8 + [-top], [hi] * 8 + [top], [lo, hi] * 4 + [top], [hi, lo] * 4 + [-top], [0] * 9, [1] + [0] * 8]
    for v in fixed[:count]:
        yield v
    for _ in range(count - len(fixed)):
        yield [rng.choice([lo, hi, rng.randint(lo, hi)]) for _ in range(8)] + [rng.randint(-top, top)]


def call(lib, op, mod, *args):
    arr = [(ctypes.c_int * 9)(*a) for a in args]
    while len(arr) < 4:
        arr.append((ctypes.c_int * 9)())
    out, canon = (ctypes.c_int * 9)(), (ctypes.c_uint * 9)()
    lib.sc_op(op, mod, *arr, out, canon)
    return list(out), list(canon)


@pytest.mark.parametrize("mod", [0, 1, 2])
@pytest.mark.parametrize("op,nargs,want", [
    (0, 2, lambda v, r: v[0] * v[1] * r), (1, 2, lambda v, r: 2 * v[0] * v[1] * r), (2, 1, lambda v, r: v[0] ** 2 * r),
    (3, 1, lambda v, r: 3 * v[0] ** 2 * r), (4, 2, lambda v, r: v[0] ** 2 * r - 2 * v[1]),
    (5, 4, lambda v, r: 2 * (v[0] * v[1] + v[2] * v[3]) * r), (6, 3, lambda v, r: (v[0] * v[1] - v[2] ** 2) * r),
    (7, 2, lambda v, r: 3 * (v[0] ** 2 - v[1] ** 2) * r), (8, 1, lambda v, r: v[0]), (9, 1, lambda v, r: v[0])])
def test_signed_ops(lib, op, nargs, want, mod):
    rng = random.Random(100 * op + mod)
    lo, hi = {7: (0, N), 8: (0, N), 9: (-3 * N, 3 * N)}.get(op, (-N, N))
    sets = [list(vectors(rng, lo, hi, 60)) for _ in range(nargs)]
    if op == 6:
        sets[1] = list(vectors(rng, -2 * N, 2 * N, 60))
    for k in range(60):
        args = [s[(k * (j + 1) + j) % 60] for j, s in enumerate(sets)] if k >= 6 else [s[k] for s in sets]
        out, canon = call(lib, op, mod, *args)
        w = want([value(a) for a in args], RINV[mod]) % P[mod]
        assert value(out) % P[mod] == w
        if op != 8:
            assert all(0 <= x <= N for x in out[:8])
        else:  # folded: within a few low-limb units of [0, 2^256)
            assert -2**229 < value(out) < 2**256 + 2**229
        if op < 8:
            assert value(canon) % P[mod] == w and value(canon) < P[mod] + P[mod] // 2**19


@pytest.mark.parametrize("mod", [0, 1])
def test_exceptional_addition_is_seen(lib, mod):
    """every H = jp within the additions' range is reported, and no random other value (values whose
    square times 2^-261 has zero low limbs, such as 2^200, may be: only two limbs are compared)"""
    def limbs(x):
        return [(x >> (29 * k)) & N for k in range(8)] + [x >> 232]
    rng = random.Random(mod)
    for j in (-3, -2, -1, 0, 1, 2, 3):
        assert lib.sc_maybe_zero(mod, (ctypes.c_int * 9)(*limbs(j * P[mod]))) == 1
        for d in (1, -1, *(rng.randrange(1, P[mod]) for _ in range(50))):
            assert lib.sc_maybe_zero(mod, (ctypes.c_int * 9)(*limbs(j * P[mod] + d))) == 0
