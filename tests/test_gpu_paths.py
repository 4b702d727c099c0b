"""Every path a plain call can take by its size: four lanes per item up to 16,384 items, one lane per
item with shared inversions above, around the sizes where the path, the workgroups or the stages'
lanes change; for message digests the order in one or three launches and one or two wavefronts to a
message. Each call holds the edge cases and corrupted generated items, repeated to the size, and every
result is compared with the oracle's."""
import hashlib

import numpy as np
import pytest

import edge_cases
import oracle_lib as O
from sigops_pkg import sigops

pytestmark = pytest.mark.gpu
SIZES = [1, 15, 16, 17, 1000, 16384, 16385, 65537]


@pytest.fixture(scope="module")
def ctx():
    c = sigops.Context()
    yield c
    c.close()


def _bytes(rows, width):
    return np.frombuffer(b"".join(rows), np.uint8).reshape(-1, width)


def _at(n, count, seed):
    """n positions in a list of count items: all of them in order (as many as fit), then random ones"""
    rng = np.random.default_rng(seed)
    return np.concatenate([np.arange(min(n, count)), rng.integers(0, count, max(0, n - count))])


@pytest.mark.parametrize("curve", [0, 1])
def test_recover_sizes(ctx, curve):
    cases = edge_cases.secp_cases(curve)
    exp = edge_cases.secp_expected(curve, cases)
    s, d, _, _ = O.gen_secp(curve, 31, 300, corrupt_ppm=200000)
    o, t = O.recover_batch(curve, s, d)
    sigs = np.concatenate([_bytes([c[1] for c in cases], 64), s])
    digs = np.concatenate([_bytes([c[2] for c in cases], 32), d])
    out = np.concatenate([_bytes([e[1] for e in exp], 64), o])
    st = np.concatenate([np.array([e[0] for e in exp], np.uint8), t])
    fn = ctx.secp256k1_recover if curve == 0 else ctx.secp256r1_recover
    for n in SIZES:
        print(f"recover curve={curve} n={n}", flush=True)
        at = _at(n, len(st), n)
        got, gst = fn(sigs[at], digs[at])
        assert np.array_equal(gst, st[at]) and np.array_equal(got, out[at]), n


@pytest.mark.parametrize("curve", [0, 1])
def test_verify_sizes(ctx, curve):
    cases = edge_cases.secp_verify_cases(curve)
    s, d, p, _ = O.gen_secp(curve, 32, 300, corrupt_ppm=200000)
    st = np.concatenate([np.array(edge_cases.secp_verify_expected(curve, cases), np.uint8),
                         O.secp_verify_batch(curve, s, d, p)])
    sigs = np.concatenate([_bytes([c[1] for c in cases], 64), s])
    digs = np.concatenate([_bytes([c[2] for c in cases], 32), d])
    pubs = np.concatenate([_bytes([c[3] for c in cases], 64), p])
    fn = ctx.secp256k1_verify if curve == 0 else ctx.secp256r1_verify
    for n in SIZES:
        print(f"verify curve={curve} n={n}", flush=True)
        at = _at(n, len(st), n)
        valid, gst = fn(sigs[at], digs[at], pubs[at])
        assert np.array_equal(gst, st[at]) and np.array_equal(valid, st[at] == 0), n


@pytest.mark.parametrize("strict", [False, True])
def test_ed25519_sizes(ctx, strict):
    # name, signature, key, message
    cases = edge_cases.ed_cases() + edge_cases.ed_strict_cases()
    oracle = O.ed25519_verify_strict if strict else O.ed25519_verify
    good = np.array([bool(oracle(c[1], c[2], c[3])) for c in cases])
    sigs, keys = [c[1] for c in cases], [c[2] for c in cases]
    msgs = [bytes(c[3]) for c in cases]
    off = np.concatenate([[0], np.cumsum(np.arange(300) * 7 % 500)]).astype(np.uint64)
    s, k, m, _ = O.gen_ed25519(33, 300, off, corrupt_ppm=200000)
    good = np.concatenate([good, (O.verify_strict_batch if strict else O.verify_batch)(s, k, m, off).astype(bool)])
    sigs = np.concatenate([_bytes(sigs, 64), s])
    keys = np.concatenate([_bytes(keys, 32), k])
    msgs += [m[int(off[i]):int(off[i + 1])].tobytes() for i in range(300)]
    lens = np.array([len(x) for x in msgs])
    for n in SIZES:
        print(f"ed25519 strict={strict} n={n}", flush=True)
        at = _at(n, len(good), n)
        moff = np.concatenate([[0], np.cumsum(lens[at])]).astype(np.uint64)
        data = np.frombuffer(b"".join(msgs[i] for i in at), np.uint8)
        valid, st = ctx.ed25519_verify(sigs[at], keys[at], data, moff, strict=strict)
        assert np.array_equal(valid, good[at]), n
        assert np.array_equal(st == 0, good[at]), n


def test_mixed_sizes(ctx):
    """mixed batches around the sizes where they change from four lanes per item to one, and from
    copying to streaming"""
    rows = []  # scheme, signature, digest or key, message, key out, status
    for curve in (0, 1):
        cases = edge_cases.secp_cases(curve)
        rows += [(curve, c[1], c[2], b"", e[1], e[0]) for c, e in zip(cases, edge_cases.secp_expected(curve, cases))]
        s, d, _, _ = O.gen_secp(curve, 41, 200, corrupt_ppm=200000)
        o, t = O.recover_batch(curve, s, d)
        rows += [(curve, s[i].tobytes(), d[i].tobytes(), b"", o[i].tobytes(), int(t[i])) for i in range(200)]
    cases = edge_cases.ed_cases()
    rows += [(2, c[1], c[2], bytes(c[3]), bytes(64), None) for c in cases]
    good = dict(zip(range(len(rows) - len(cases), len(rows)), edge_cases.ed_expected(cases)))
    off = np.concatenate([[0], np.cumsum(np.arange(200) * 41 % 4200)]).astype(np.uint64)
    s, k, m, _ = O.gen_ed25519(43, 200, off, corrupt_ppm=200000)
    ok = O.verify_batch(s, k, m, off)
    for i in range(200):
        good[len(rows)] = bool(ok[i])
        rows.append((2, s[i].tobytes(), k[i].tobytes(), m[int(off[i]):int(off[i + 1])].tobytes(), bytes(64), None))
    schemes = np.array([r[0] for r in rows], np.uint8)
    sigs, aux, out = (_bytes([r[j] for r in rows], w) for j, w in ((1, 64), (2, 32), (4, 64)))
    lens = np.array([len(r[3]) for r in rows])
    perm = np.random.default_rng(5).permutation(len(rows))
    for n in (1, 15, 17, len(rows), 16384, 24576, 24577, 65536, 262143, 262144):
        print(f"mixed n={n}", flush=True)
        at = perm[_at(n, len(rows), n)]
        moff = np.concatenate([[0], np.cumsum(lens[at])]).astype(np.uint64)
        data = np.frombuffer(b"".join(rows[i][3] for i in at), np.uint8)
        got, st = ctx.batch(schemes[at], sigs[at], aux[at], data, moff)
        assert np.array_equal(got, out[at]), n
        for j in range(len(rows)):
            want = rows[j][5]
            mine = st[at == j]
            assert np.all((mine == 0) == good[j]) if want is None else np.all(mine == want), (n, j)


# one length (two wavefronts to a message while all lanes are not filled, one wavefront above), lengths
# around the blocks' edges, and long ones among short ones
@pytest.mark.parametrize("lens", [[40], [0, 1, 55, 56, 63, 64, 119, 120, 3, 200], [5] * 40 + [4096, 4300, 700]])
@pytest.mark.parametrize("skew", [0, 4])
def test_message_new_sizes(ctx, lens, skew):
    import torch
    for n in [1, 64, 65, 8192, 8193, 40001, 300001]:
        if n * np.mean(lens) > 4e7:
            continue
        print(f"message_new lens={lens[-1]} skew={skew} n={n}", flush=True)
        rng = np.random.default_rng(n)
        ln = np.array(lens)[_at(n, len(lens), n)]
        rng.shuffle(ln)
        off = np.concatenate([[0], np.cumsum(ln)]).astype(np.int64)
        buf = rng.integers(0, 256, skew + int(off[-1]) + 16, dtype=np.uint8)
        want = [hashlib.sha256(buf[skew + off[i]:skew + off[i + 1]]).digest() for i in range(n)]
        d_buf, d_off = torch.from_numpy(buf).cuda(), torch.from_numpy(off).cuda()
        d_out = torch.zeros(n, 32, dtype=torch.uint8, device="cuda")
        ctx.message_new_dev(d_buf.data_ptr() + skew, d_off.data_ptr(), n, d_out.data_ptr())
        torch.cuda.synchronize()
        assert np.array_equal(d_out.cpu().numpy(), _bytes(want, 32)), n


@pytest.mark.parametrize("order", [0, 1, 2])
def test_mixed_bucket_orders(order):
    """tiles shared by neighbouring Ed25519 buckets and first tiles by place, in every bucket order, with
    one and two workgroups per compute unit: keys and statuses as in the items' own order"""
    for blocks in (1, 2):
        c = sigops.Context(bucket_order=order, blocks_per_cu=blocks)
        n = 30011
        s0, d0, p0, _ = O.gen_secp(0, 51, 100, corrupt_ppm=0)
        s1, d1, p1, _ = O.gen_secp(1, 52, 100, corrupt_ppm=0)
        off = np.concatenate([[0], np.cumsum(np.arange(300) * 29 % 5000)]).astype(np.uint64)
        s2, k2, m2, _ = O.gen_ed25519(53, 300, off, corrupt_ppm=300000)
        ok = np.concatenate([np.ones(200, bool), O.verify_batch(s2, k2, m2, off).astype(bool)])
        sigs, aux = np.concatenate([s0, s1, s2]), np.concatenate([d0, d1, k2])
        keys = np.concatenate([p0, p1, np.zeros((300, 64), np.uint8)])
        lens = np.concatenate([np.zeros(200, np.int64), np.diff(off.astype(np.int64))])
        begin = np.concatenate([np.zeros(200, np.int64), off[:-1].astype(np.int64)])
        at = np.random.default_rng(order).integers(0, 500, n)
        moff = np.concatenate([[0], np.cumsum(lens[at])]).astype(np.uint64)
        data = np.concatenate([m2[begin[i]:begin[i] + lens[i]] for i in at])
        schemes = np.where(at < 100, 0, np.where(at < 200, 1, 2)).astype(np.uint8)
        print(f"mixed order={order} blocks={blocks}", flush=True)
        c.set_streaming(False)
        got, st = c.batch(schemes, sigs[at], aux[at], data, moff)
        c.close()
        assert np.array_equal(st == 0, ok[at]) and np.array_equal(got, keys[at])
