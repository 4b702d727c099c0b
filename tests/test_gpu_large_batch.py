"""Mixed batches above the sizes that run on four lanes per item (24,576 items): the bucketed launches with
placed tiles and shared inversions. Items are drawn, with repetition, from a set of edge cases and corrupted
generated ones, so every result is compared with the oracle's."""
import numpy as np
import pytest
import torch

import edge_cases
import oracle_lib as O
from sigops_pkg import sigops

pytestmark = pytest.mark.gpu


class Rows:
    """distinct items: scheme, signature, digest or key, message, and the oracle's key and verdict (the status
    of a secp item; for Ed25519 only whether it is 0)"""

    def __init__(self):
        rows = []
        for curve in (0, 1):
            cases = edge_cases.secp_cases(curve)
            rows += [(curve, c[1], c[2], b"", e[1], e[0]) for c, e in
                     zip(cases, edge_cases.secp_expected(curve, cases))]
            s, d, _, _ = O.gen_secp(curve, 61, 200, corrupt_ppm=200000)
            o, t = O.recover_batch(curve, s, d)
            rows += [(curve, s[i].tobytes(), d[i].tobytes(), b"", o[i].tobytes(), int(t[i])) for i in range(200)]
        cases = edge_cases.ed_cases()
        rows += [(2, c[1], c[2], bytes(c[3]), bytes(64), 0 if e else 1) for c, e in
                 zip(cases, edge_cases.ed_expected(cases))]
        off = np.concatenate([[0], np.cumsum(np.arange(200) * 37 % 5200)]).astype(np.uint64)
        s, k, m, _ = O.gen_ed25519(63, 200, off, corrupt_ppm=200000)
        ok = O.verify_batch(s, k, m, off)
        rows += [(2, s[i].tobytes(), k[i].tobytes(), m[int(off[i]):int(off[i + 1])].tobytes(), bytes(64),
                  0 if ok[i] else 1) for i in range(200)]
        col = [list(c) for c in zip(*rows)]
        self.scheme = np.array(col[0], np.uint8)
        self.sig, self.aux, self.out = (np.frombuffer(b"".join(col[j]), np.uint8).reshape(-1, w)
                                        for j, w in ((1, 64), (2, 32), (4, 64)))
        self.lens = np.array([len(x) for x in col[3]], np.int64)
        self.begin = np.concatenate([[0], np.cumsum(self.lens)[:-1]])
        self.msgs = np.frombuffer(b"".join(col[3]) + bytes(16), np.uint8)
        self.verdict = np.array(col[5], np.uint8)

    def draw(self, n, seed, longest=1 << 30):
        """a batch of n items (messages of at most `longest` bytes): its arrays, and the rows they are"""
        rng = np.random.default_rng(seed)
        at = rng.choice(np.flatnonzero(self.lens <= longest), n)
        lens = self.lens[at]
        off = np.concatenate([[0], np.cumsum(lens)])
        data = self.msgs[np.repeat(self.begin[at] - off[:-1], lens) + np.arange(off[-1])]
        return (self.scheme[at], self.sig[at], self.aux[at], data, off.astype(np.uint64)), at

    def check(self, at, out, st, what):
        assert np.array_equal(out, self.out[at]), what
        verdict = np.where(self.scheme[at] == 2, st != 0, st)
        assert np.array_equal(verdict, self.verdict[at]), what


@pytest.fixture(scope="module")
def rows():
    return Rows()


def test_plain_calls_where_inversions_are_shared():
    """plain recoveries and verifications around the size from which they share inversions between items
    (three and four items to a lane), edge cases and corrupted items among the shared ones"""
    ctx = sigops.Context()
    for curve in (0, 1):
        cases = edge_cases.secp_cases(curve)
        exp = edge_cases.secp_expected(curve, cases)
        s, d, p, _ = O.gen_secp(curve, 71, 300, corrupt_ppm=200000)
        o, t = O.recover_batch(curve, s, d)
        sigs = np.concatenate([np.frombuffer(b"".join(c[1] for c in cases), np.uint8).reshape(-1, 64), s])
        digs = np.concatenate([np.frombuffer(b"".join(c[2] for c in cases), np.uint8).reshape(-1, 32), d])
        out = np.concatenate([np.frombuffer(b"".join(e[1] for e in exp), np.uint8).reshape(-1, 64), o])
        st = np.concatenate([np.array([e[0] for e in exp], np.uint8), t])
        vcases = edge_cases.secp_verify_cases(curve)
        vst = np.concatenate([np.array(edge_cases.secp_verify_expected(curve, vcases), np.uint8),
                              O.secp_verify_batch(curve, s, d, p)])
        vsigs = np.concatenate([np.frombuffer(b"".join(c[1] for c in vcases), np.uint8).reshape(-1, 64), s])
        vdigs = np.concatenate([np.frombuffer(b"".join(c[2] for c in vcases), np.uint8).reshape(-1, 32), d])
        vpubs = np.concatenate([np.frombuffer(b"".join(c[3] for c in vcases), np.uint8).reshape(-1, 64), p])
        for n in (131072, 196607, 196608, 200003):
            print(f"shared inversions curve={curve} n={n}", flush=True)
            at = np.random.default_rng(n).integers(0, len(st), n)
            got, gst = (ctx.secp256k1_recover if curve == 0 else ctx.secp256r1_recover)(sigs[at], digs[at])
            assert np.array_equal(gst, st[at]) and np.array_equal(got, out[at]), n
            at = np.random.default_rng(n).integers(0, len(vst), n)
            _, gst = (ctx.secp256k1_verify if curve == 0 else ctx.secp256r1_verify)(vsigs[at], vdigs[at], vpubs[at])
            assert np.array_equal(gst, vst[at]), n
    ctx.close()


def _on_device(batch):
    sch, sig, aux, data, off = batch
    data = np.concatenate([data, np.zeros(32 - len(data) % 16, np.uint8)])
    n = len(sch)
    return ([torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in (sch, sig, aux, data, off.astype(np.int64))], n,
            torch.zeros(n, 64, dtype=torch.uint8, device="cuda"), torch.full((n,), 0xEE, dtype=torch.uint8, device="cuda"))


def _enqueue(ctx, dev, stream):
    ins, n, out, st = dev
    ctx.batch_dev(*[t.data_ptr() for t in ins], n, out.data_ptr(), st.data_ptr(), stream)


def test_two_contexts_at_once(rows):
    """batches of two contexts on two streams, together more than the GPU holds at a time: the workgroups of one
    wait for the other's, and their first tiles go to the wavefronts that run"""
    ctxs = [sigops.Context(), sigops.Context()]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    sizes = [(60000, 60011), (130000, 24576), (24577, 100003)]
    drawn = [[rows.draw(n, 10 * k + j) for j, n in enumerate(pair)] for k, pair in enumerate(sizes)]
    dev = [[_on_device(b) for b, _ in pair] for pair in drawn]
    torch.cuda.synchronize()
    print("two contexts", sizes, flush=True)
    for _ in range(2):
        for pair in dev:
            for j in range(2):
                _enqueue(ctxs[j], pair[j], streams[j].cuda_stream)
    torch.cuda.synchronize()
    for pair, d in zip(drawn, dev):
        for (_, at), (_, n, out, st) in zip(pair, d):
            rows.check(at, out.cpu().numpy(), st.cpu().numpy(), n)
    for c in ctxs:
        c.close()


def test_sizes_where_the_launch_changes(rows):
    """around the sizes where a batch goes from four lanes per item to one, from tiles by counter to tiles by
    place, and to shared inversions; host calls copied, and the largest two on the device"""
    ctx = sigops.Context()
    ctx.set_streaming(False)
    for n in (20480, 20481, 32768, 33011, 65536, 65537, 131072):
        print(f"mixed n={n}", flush=True)
        batch, at = rows.draw(n, n)
        rows.check(at, *ctx.batch(*batch), n)
    for n in (786431, 786432):
        print(f"mixed n={n}", flush=True)
        batch, at = rows.draw(n, n, longest=300)
        dev = _on_device(batch)
        _enqueue(ctx, dev, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        rows.check(at, dev[2].cpu().numpy(), dev[3].cpu().numpy(), n)
    ctx.close()


def test_calls_in_pieces(rows):
    """device calls of more than 2^22 items run in pieces of that size: results of ragged last pieces (1, 15
    and 17 items and a larger one), and stage timing that covers every piece"""
    piece = 1 << 22
    ctx = sigops.Context(max_batch=piece + 30011)
    s = torch.cuda.current_stream().cuda_stream
    secp = [np.flatnonzero(rows.scheme == c) for c in (0, 1)]
    cases = edge_cases.secp_verify_cases(1)
    vst = np.array(edge_cases.secp_verify_expected(1, cases), np.uint8)
    vcol = [torch.from_numpy(np.frombuffer(b"".join(c[j] for c in cases), np.uint8).reshape(len(cases), -1).copy()).cuda()
            for j in (1, 2, 3)]
    for curve, tail in ((0, 1), (1, 15), (1, 17), (0, 30011)):
        n = piece + tail
        print(f"pieces n={n}", flush=True)
        out = torch.zeros(n, 64, dtype=torch.uint8, device="cuda")
        st = torch.full((n,), 0xEE, dtype=torch.uint8, device="cuda")
        at = torch.from_numpy(np.random.default_rng(tail).choice(secp[curve], n)).cuda()
        sig, aux, want = (torch.from_numpy(x.copy()).cuda() for x in (rows.sig, rows.aux, rows.out))
        sig, aux = sig[at], aux[at]
        ctx.secp_recover_dev(curve, sig.data_ptr(), aux.data_ptr(), n, out.data_ptr(), st.data_ptr(), s)
        torch.cuda.synchronize()
        assert torch.equal(st, torch.from_numpy(rows.verdict).cuda()[at]) and torch.equal(out, want[at]), n
        at = torch.from_numpy(np.random.default_rng(tail).integers(0, len(cases), n)).cuda()
        v = [x[at] for x in vcol]
        ctx.secp256r1_verify_dev(v[0].data_ptr(), v[1].data_ptr(), v[2].data_ptr(), n, st.data_ptr(), s)
        torch.cuda.synchronize()
        assert torch.equal(st, torch.from_numpy(vst).cuda()[at]), n
        batch, at = rows.draw(n, tail, longest=60)
        dev = _on_device(batch)
        _enqueue(ctx, dev, s)
        torch.cuda.synchronize()
        rows.check(at, dev[2].cpu().numpy(), dev[3].cpu().numpy(), n)
    # the larger piece is 140 times the last one, and so is its time
    ctx.set_stage_timing(True)
    _enqueue(ctx, dev, s)
    whole = ctx.batch_stage_ms()["verify_kernel"]
    ins, n, out, st = dev
    _enqueue(ctx, (ins, tail, out, st), s)
    part = ctx.batch_stage_ms()["verify_kernel"]
    print(f"stage timing: {whole:.2f} ms, the last piece's items alone {part:.2f} ms", flush=True)
    assert whole > 4 * part
    ctx.close()


def _rounds(ctx, rows, sizes, what):
    for n in sizes:
        print(f"{what} n={n}", flush=True)
        batch, at = rows.draw(n, n, longest=300 if n > 200000 else 1 << 30)
        dev = _on_device(batch)
        _enqueue(ctx, dev, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        rows.check(at, dev[2].cpu().numpy(), dev[3].cpu().numpy(), (what, n))


@pytest.mark.parametrize("order", [0, 1, 2])
def test_tile_rounds(rows, order):
    """tiles of 64 to 256 items in every bucket order, Ed25519 items of 1 to 40 blocks sharing them: tiles by
    counter, by place and with shared inversions"""
    for rounds in (1, 2, 3, 4):
        ctx = sigops.Context(tuned=False, tile_rounds=rounds, bucket_order=order)
        _rounds(ctx, rows, [25013, 70001, 200017] + ([786433] if rounds == 1 + order else []),
                f"rounds={rounds} order={order}")
        ctx.close()


def test_one_wave_per_simd(rows):
    """the persistent kernel built for one wavefront per SIMD shares inversions at every size"""
    ctx = sigops.Context(tuned=False, waves=1)
    _rounds(ctx, rows, [20481, 25013, 100003], "waves=1")
    ctx.close()


def test_graph_eager_and_timed_launches(rows):
    """calls of every form in turn on one context, replayed from its graphs, launched eagerly and timed: on
    four lanes per item, in one kernel, with shared inversions"""
    sizes = (3000, 30011, 786433)
    drawn = [rows.draw(n, n, longest=300) for n in sizes]
    dev = [_on_device(b) for b, _ in drawn]
    stream = torch.cuda.current_stream().cuda_stream
    graph, eager = sigops.Context(), sigops.Context(use_graph=False)
    for rep in range(3):
        for ctx, timed in ((graph, False), (eager, False), (graph, True)):
            ctx.set_stage_timing(timed)
            for (_, at), d in zip(drawn, dev):
                print(f"launch forms rep={rep} eager={ctx is eager} timed={timed} n={d[1]}", flush=True)
                d[2].zero_()
                d[3].fill_(0xEE)
                _enqueue(ctx, d, stream)
                if timed:
                    ms = ctx.batch_stage_ms()
                    assert all(v >= 0 for v in ms.values()) and ms["verify_kernel"] > 0
                torch.cuda.synchronize()
                rows.check(at, d[2].cpu().numpy(), d[3].cpu().numpy(), (rep, timed, d[1]))
            ctx.set_stage_timing(False)
    graph.close()
    eager.close()


def test_calls_in_a_captured_graph(rows):
    """calls of every form recorded into the caller's own graph, on a context that has run only one of them:
    every replay, with eager calls on the same context between them, gives the oracle's results"""
    ctx = sigops.Context()
    s = torch.cuda.Stream()
    warm, warm_at = rows.draw(1000, 1)
    warm = _on_device(warm)
    _enqueue(ctx, warm, s.cuda_stream)
    torch.cuda.synchronize()
    for n in (1000, 30011, 786433):
        print(f"captured call n={n}", flush=True)
        batch, at = rows.draw(n, n, longest=300)
        dev = _on_device(batch)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            _enqueue(ctx, dev, s.cuda_stream)
        for replay in range(4):
            dev[2].zero_()
            dev[3].fill_(0xEE)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            rows.check(at, dev[2].cpu().numpy(), dev[3].cpu().numpy(), (n, replay))
            warm[3].fill_(0xEE)
            _enqueue(ctx, warm, torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            rows.check(warm_at, warm[2].cpu().numpy(), warm[3].cpu().numpy(), (n, replay))
        del graph
    ctx.close()
