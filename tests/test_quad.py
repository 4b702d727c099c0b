"""Four-lane point formulas (csrc/quad.hpp), host build, against affine arithmetic on Python integers:
programs of doublings, additions and subtractions, and the exceptional additions."""
import ctypes
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "wgpu-sigops_amd", "csrc")
CURVES = [  # p, a, b, generator
    (2**256 - 2**32 - 977, 0, 7,
     (0x79BE667EF9DCBBAC55A06295CE870B07029BFCDB2DCE28D959F2815B16F81798,
      0x483ADA7726A3C4655DA4FBFC0E1108A8FD17B448A68554199C47D08FFB10D4B8)),
    (2**256 - 2**224 + 2**192 + 2**96 - 1, -3, 0x5AC635D8AA3A93E7B3EBBD55769886BC651D06B0CC53B0F63BCE3C3E27D2604B,
     (0x6B17D1F2E12C4247F8BCE6E563A440F277037D812DEB33A0F4A13945D898C296,
      0x4FE342E2FE1A7F9B8EE7EB4A7C0F9E162BCE33576B315ECECBB6406837BF51F5))]
PED = 2**255 - 19
DED = -121665 * pow(121666, -1, PED) % PED
BED = (15112221349535400772501151409588531511454012693041857206046113283949847762202,
       4 * pow(5, -1, PED) % PED)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("quad") / "libquad.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-DSIGOPS_HOST_CHECK=1",
                    "-I" + CSRC, "-o", so, os.path.join(HERE, "devcheck", "quad_check.cpp")], check=True)
    return ctypes.CDLL(so)


def add(curve, P, Q):
    p, a, _, _ = CURVES[curve]
    if P == Q:
        m = (3 * P[0] ** 2 + a) * pow(2 * P[1], -1, p)
    else:
        m = (Q[1] - P[1]) * pow(Q[0] - P[0], -1, p)
    x = (m * m - P[0] - Q[0]) % p
    return x, (m * (P[0] - x) - P[1]) % p


def mul(curve, k, P):
    R = None
    for b in bin(k)[2:]:
        R = add(curve, R, R) if R else None
        if b == "1":
            R = add(curve, R, P) if R else P
    return R


def enc(P):
    return P[0].to_bytes(32, "big") + P[1].to_bytes(32, "big")


PROGRAMS = ["a", "s", "d", "da", "ds", "dddda", "ddddas" * 3, "aaaa", "dddd" * 8, "d" * 40 + "a" * 20 + "s" * 7]


@pytest.mark.parametrize("curve", [0, 1])
@pytest.mark.parametrize("prog", PROGRAMS)
def test_secp_programs(lib, curve, prog):
    p, _, _, G = CURVES[curve]
    rng = random.Random(prog + str(curve))
    for _ in range(6):
        P, Q = mul(curve, rng.randrange(2, 2**255), G), mul(curve, rng.randrange(2, 2**255), G)
        out = ctypes.create_string_buffer(64)
        assert lib.qc_secp(curve, prog.encode(), enc(P), enc(Q), out) == 0
        for c in prog:
            P = add(curve, P, P) if c == "d" else add(curve, P, Q if c == "a" else (Q[0], p - Q[1]))
        assert int.from_bytes(out.raw[:32], "big") == P[0]
        assert int.from_bytes(out.raw[32:], "big") == 2 * P[1] % p


@pytest.mark.parametrize("curve", [0, 1])
def test_secp_exceptional_additions(lib, curve):
    G = CURVES[curve][3]
    P = mul(curve, 12345, G)
    out = ctypes.create_string_buffer(64)
    for prog, Q in (("a", P), ("s", P), ("da", mul(curve, 2 * 12345, G)), ("dds", mul(curve, 4 * 12345, G))):
        assert lib.qc_secp(curve, prog.encode(), enc(P), enc(Q), out) == 1


def ed_add(P, Q):
    x1, y1, x2, y2 = *P, *Q
    k = DED * x1 * x2 * y1 * y2
    return ((x1 * y2 + x2 * y1) * pow(1 + k, -1, PED) % PED, (y1 * y2 + x1 * x2) * pow(1 - k, -1, PED) % PED)


@pytest.mark.parametrize("prog", PROGRAMS)
def test_edwards_programs(lib, prog):
    rng = random.Random(prog)
    pts = [(0, 1), (0, PED - 1), BED]  # the identity and the point of order 2 among them: complete formulas
    for _ in range(4):
        pts.append(ed_add(pts[-1], pts[rng.randrange(2, len(pts))]))
    for P in pts:
        for Q in pts:
            out = ctypes.create_string_buffer(64)
            lib.qc_ed(prog.encode(), enc(P), enc(Q), out)
            R = P
            for c in prog:
                R = ed_add(R, R) if c == "d" else ed_add(R, Q if c == "a" else ((PED - Q[0]) % PED, Q[1]))
            assert (int.from_bytes(out.raw[:32], "big"), int.from_bytes(out.raw[32:], "big")) == R
