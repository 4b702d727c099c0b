"""What the kernels run by default, built for the host with the bound checker on (tests/devcheck/wide_check.cpp):
the ladders with the wide fixed-base tables item by item, through the stages that share inversions, and on the
four lanes of a quad. The tables' entries are computed here with Python integers."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import edge_cases
import oracle_lib as O
import pyref

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "wgpu-sigops_amd", "csrc")
R = 1 << 261  # Montgomery form
PENDING = 0xFF
ENTRY = ctypes.CFUNCTYPE(None, ctypes.c_int, ctypes.c_int, ctypes.c_uint, ctypes.POINTER(ctypes.c_uint32))
_windows = {}  # (curve, window) -> 2^(16 window) G
_entries = {}


def _window(curve, i):
    if (curve, i) not in _windows:
        k = 1 << (16 * i)
        _windows[curve, i] = (pyref.e_mul(_base(), k) if curve == 2 else
                              pyref.w_mul(pyref.CURVES[curve], pyref.CURVES[curve]["G"], k))
    return _windows[curve, i]


def _base():
    return pyref.e_decompress((4 * pow(5, -1, pyref.EP) % pyref.EP).to_bytes(32, "little"))


def _entry(curve, i, j):
    """the values of entry j, (2j + 1) 2^(16 i) G: x and 2y, or (y + x)/2, (y - x)/2 and dxy"""
    if (curve, i, j) not in _entries:
        if curve == 2:
            x, y = pyref.e_mul(_window(2, i), 2 * j + 1)[:2]
            p, h = pyref.EP, pow(2, -1, pyref.EP)
            d = -121665 * pow(121666, -1, p)
            vals = ((y + x) * h, (y - x) * h, d * x * y)
        else:
            p = pyref.CURVES[curve]["p"]
            x, y = pyref.w_mul(pyref.CURVES[curve], _window(curve, i), 2 * j + 1)
            vals = (x, 2 * y)
        _entries[curve, i, j] = [(v * R % p >> (32 * k)) & 0xFFFFFFFF for v in vals for k in range(8)]
    return _entries[curve, i, j]


def _fill(curve, i, j, out):
    for k, w in enumerate(_entry(curve, i, j)):
        out[k] = w


_callback = ENTRY(_fill)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("wide") / "libwide.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-DSIGOPS_HOST_CHECK=1",
                    "-I" + CSRC, "-o", so, os.path.join(HERE, "devcheck", "wide_check.cpp")], check=True)
    L = ctypes.CDLL(so)
    L.wc_entries(_callback)
    return L


def _secp_items(curve):
    """signatures, digests, and the expected status and key of each"""
    cases = edge_cases.secp_cases(curve)
    s, d, _, _ = O.gen_secp(curve, 81, 40, corrupt_ppm=150000)
    o, t = O.recover_batch(curve, s, d)
    exp = edge_cases.secp_expected(curve, cases)
    return ([c[1] for c in cases] + [x.tobytes() for x in s], [c[2] for c in cases] + [x.tobytes() for x in d],
            [(e[0], e[1]) for e in exp] + [(int(a), b.tobytes()) for a, b in zip(t, o)])


@pytest.mark.parametrize("quad", [0, 1])
@pytest.mark.parametrize("curve", [0, 1])
def test_recover(lib, curve, quad):
    careful = 0
    for sig, dig, exp in zip(*_secp_items(curve)):
        out = ctypes.create_string_buffer(64)
        st = lib.wc_recover(curve, sig, dig, out, quad)
        careful += st >> 8
        assert ((st & 0xFF), out.raw) == exp, (sig.hex(), dig.hex())
    assert careful > 0  # exceptional additions were among them


@pytest.mark.parametrize("curve", [0, 1])
def test_exceptional_additions_in_the_table_part(lib, curve):
    """u2 R = +-(the entry of u1's lowest digit): the first addition after the ladder doubles or meets its
    negative; and the same at the last one, where the sum of the others is the entry of the top digit"""
    c = pyref.CURVES[curve]
    n = c["n"]
    hits = 0
    for m in (1, 3, 12345, 65535):
        for u1 in (m, n - m, m + (7 << 16), n - m - (7 << 16) & ~1 | 1, 2 * m):
            for quad in (0, 1):
                Rm = pyref.w_mul(c, c["G"], m)
                r = Rm[0] % n
                if r != Rm[0]:
                    continue
                s, odd = r, Rm[1] & 1  # u2 = 1
                sig = edge_cases._enc_sig(curve, r, s, odd)
                dig = (-u1 * r % n).to_bytes(32, "big")
                out = ctypes.create_string_buffer(64)
                st = lib.wc_recover(curve, sig, dig, out, quad)
                hits += st >> 8
                assert (st & 0xFF, out.raw) == pyref.secp_recover(curve, sig, dig), (m, u1, quad)
    assert hits >= 8


@pytest.mark.parametrize("curve", [0, 1])
def test_verify(lib, curve):
    cases = edge_cases.secp_verify_cases(curve)
    s, d, p, _ = O.gen_secp(curve, 82, 30, corrupt_ppm=150000)
    exp = list(edge_cases.secp_verify_expected(curve, cases)) + [int(x) for x in O.secp_verify_batch(curve, s, d, p)]
    items = [c[1:4] for c in cases] + [(a.tobytes(), b.tobytes(), q.tobytes()) for a, b, q in zip(s, d, p)]
    for (sig, dig, pub), e in zip(items, exp):
        assert lib.wc_verify(curve, sig, dig, pub) & 0xFF == e, (sig.hex(), dig.hex())


@pytest.mark.parametrize("lanes", [1, 3, 16])
@pytest.mark.parametrize("curve", [0, 1])
def test_shared_inversions(lib, curve, lanes):
    """items of every kind, and positions that hold none, in one inversion"""
    sigs, digs, exp = _secp_items(curve)
    rng = np.random.default_rng(curve)
    for positions in (1, lanes, lanes + 1, 90):
        at = rng.integers(0, len(sigs), positions).astype(np.uint32)
        at = np.where(rng.random(positions) < 0.2, np.uint32(0xFFFFFFFF), at).astype(np.uint32)
        # one position per item: results are written by item
        _, first = np.unique(at, return_index=True)
        keep = np.zeros(positions, bool)
        keep[first] = True
        at[~keep] = 0xFFFFFFFF
        out, st = np.full((len(sigs), 64), 0x77, np.uint8), np.full(len(sigs), 0x77, np.uint8)
        lib.wc_stages(curve, 0, positions, at.ctypes.data_as(ctypes.c_void_p), lanes, b"".join(sigs), b"".join(digs),
                      None, out.ctypes.data_as(ctypes.c_void_p), st.ctypes.data_as(ctypes.c_void_p))
        for i in range(len(sigs)):
            if i not in at:
                assert st[i] == 0x77 and np.all(out[i] == 0x77)
            elif st[i] == PENDING:
                assert not out[i].any()
            else:
                assert (int(st[i]), out[i].tobytes()) == exp[i], i
    cases = edge_cases.secp_verify_cases(curve)
    want = edge_cases.secp_verify_expected(curve, cases)
    at, st = rng.permutation(len(cases)).astype(np.uint32), np.zeros(len(cases), np.uint8)
    lib.wc_stages(curve, 1, len(cases), at.ctypes.data_as(ctypes.c_void_p), lanes, b"".join(c[1] for c in cases),
                  b"".join(c[2] for c in cases), b"".join(c[3] for c in cases), None,
                  st.ctypes.data_as(ctypes.c_void_p))
    assert all(s in (PENDING, w) for s, w in zip(st, want))
    assert 0 < np.count_nonzero(st == PENDING) < len(cases) // 2


@pytest.mark.parametrize("quad", [0, 2])
@pytest.mark.parametrize("strict", [0, 1])
def test_ed25519(lib, strict, quad):
    cases = edge_cases.ed_cases() + (edge_cases.ed_strict_cases() if strict else [])
    oracle = O.ed25519_verify_strict if strict else O.ed25519_verify
    for _, sig, pk, m in cases:
        assert (lib.wc_ed25519(sig, pk, bytes(m), len(m), strict | quad) == 0) == bool(oracle(sig, pk, m))
    off = np.concatenate([[0], np.cumsum(np.arange(40) * 13 % 300)]).astype(np.uint64)
    s, k, m, bad = O.gen_ed25519(83, 40, off, corrupt_ppm=200000)
    for i in range(40):
        msg = m[int(off[i]):int(off[i + 1])].tobytes()
        assert (lib.wc_ed25519(s[i].tobytes(), k[i].tobytes(), msg, len(msg), strict | quad) == 0) == (not bad[i])
