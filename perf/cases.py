"""The work this library is measured on: calls a user's program makes, through the public entry
points, over the sizes they are made at.

A case is a dict of plain values. ``kind`` names the entry point, ``where`` where the caller's data
lives (``host``: numpy arrays in and out, transfers included; ``device``: tensors resident in HBM),
``n`` the number of items, ``corrupt`` the corrupted items per million and ``max_len`` the longest
message. Signatures come from the library's seeded device generator (valid fuel-format signatures,
some with one bit flipped), message lengths from numpy: all of it a function of the seed.

Outputs are keys, addresses, digests and status bytes: whole bytes, equal or wrong.
"""
import hashlib
import importlib

import numpy as np
import torch

sigops = importlib.import_module("wgpu-sigops_amd")

MIX = (0.5, 0.3, 0.2)  # secp256k1, secp256r1, Ed25519: the mixed workload of the benchmark

# kind -> (smallest, largest) n of the range the listed cases stand for
RANGES = {
    "recover": (1, 1 << 19),
    "address": (1, 1 << 17),
    "verify": (1, 1 << 17),
    "ed25519": (1, 1 << 17),
    "ed25519_strict": (1, 1 << 17),
    "mixed": (3, 1 << 20),
    "digests": (1, 1 << 19),
    "serve": (2, 64),
}


def listed():
    return [
        # a node checking the few transactions that have just arrived: latency and launches count
        dict(name="k1_recover_host_16", kind="recover", curve=0, where="host", n=16, corrupt=0),
        # the reference benchmark's smallest batch, host to host
        dict(name="k1_recover_host_1024", kind="recover", curve=0, where="host", n=1024, corrupt=0),
        # passkey signatures of a block range, host to host (benchmark configuration)
        dict(name="r1_recover_host_65536", kind="recover", curve=1, where="host", n=65536, corrupt=0),
        # attestations with payloads up to 1 KB, a tenth of them bad (benchmark configuration)
        dict(name="ed25519_host_65536", kind="ed25519", where="host", n=65536, corrupt=100000, max_len=1024,
             log_lengths=False),
        # chain re-validation with the data already on the GPU: the largest plain recovery
        dict(name="k1_recover_device_524288", kind="recover", curve=0, where="device", n=1 << 19, corrupt=50000),
        # the headline: one batch of the three schemes, resident, messages up to 4 KB
        dict(name="mixed_device_1048576", kind="mixed", where="device", n=1 << 20, corrupt=50000, max_len=4096),
        # the same mix as a service's ordinary batch, host to host, a ragged size
        dict(name="mixed_host_100003", kind="mixed", where="host", n=100003, corrupt=50000, max_len=4096),
        # known-key verification of one ordinary block, resident, an odd size
        dict(name="r1_verify_device_20011", kind="verify", curve=1, where="device", n=20011, corrupt=50000),
        # recovery straight to addresses, host to host, an odd size
        dict(name="k1_address_host_5003", kind="address", curve=0, where="host", n=5003, corrupt=20000),
        # a validator set's votes: a few hundred strict verifications of short messages
        dict(name="ed25519_strict_device_300", kind="ed25519_strict", where="device", n=300, corrupt=20000, max_len=200,
             log_lengths=False),
        # digests of transactions of every length, the step before recovery
        dict(name="digests_device_209715", kind="digests", where="device", n=209715, max_len=4096),
        # the request server under a burst: requests of 1..4096 mixed items, all waited for
        dict(name="serve_burst_24", kind="serve", n=24, corrupt=50000, max_len=4096),
    ]


def draw(rng):
    kind = rng.choice(sorted(RANGES))
    lo, hi = RANGES[kind]
    n = int(round(lo * (hi / lo) ** rng.random()))
    if n > 8 and rng.random() < 0.7:
        n |= 1
    n = max(lo, min(n, hi))
    case = dict(kind=kind, n=n)
    if kind != "serve":
        case["where"] = rng.choice(["host", "device"]) if kind not in ("address", "digests") else (
            "host" if kind == "address" else "device")
    if kind in ("recover", "address", "verify"):
        case["curve"] = rng.choice([0, 1])
    if kind != "digests":
        case["corrupt"] = rng.choice([0, 20000, 50000, 100000])
    if kind in ("ed25519", "ed25519_strict"):
        case["max_len"] = rng.choice([0, 32, 200, 1024, 4096])
        case["log_lengths"] = rng.random() < 0.5
    elif kind in ("mixed", "digests", "serve"):
        case["max_len"] = rng.choice([200, 1024, 4096])
    return case


# ---- inputs ----

def _lengths(rng, n, max_len, log):
    if not log:
        return rng.integers(0, max_len + 1, n)
    return (np.floor(np.exp(rng.random(n) * np.log(max_len + 1))) - 1).astype(np.int64).clip(0, max_len)


def _offsets(lens):
    off = np.zeros(len(lens) + 1, np.int64)
    np.cumsum(lens, out=off[1:])
    return off


def _bytes(n, width):
    return torch.empty((n, width) if width else n, dtype=torch.uint8, device="cuda")


def _message_buffer(total):
    # 4-byte aligned and readable past the last message, as the device entry points ask
    return torch.zeros((total + 16 + 15) // 16 * 16, dtype=torch.uint8, device="cuda")


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _gen_secp(ctx, curve, n, seed, corrupt):
    sigs, digests, keys = _bytes(n, 64), _bytes(n, 32), _bytes(n, 64)
    ctx.gen_secp_dev(curve, seed, n, corrupt, sigs.data_ptr(), digests.data_ptr(), keys.data_ptr(), None, _stream())
    return sigs, digests, keys


def _gen_ed25519(ctx, lens, seed, corrupt):
    n = len(lens)
    off = torch.from_numpy(_offsets(lens)).cuda()
    msgs = _message_buffer(int(lens.sum()))
    sigs, keys = _bytes(n, 64), _bytes(n, 32)
    ctx.gen_ed25519_dev(seed, n, corrupt, off.data_ptr(), msgs.data_ptr(), sigs.data_ptr(), keys.data_ptr(), None,
                        _stream())
    return sigs, keys, msgs, off


def _gen_mixed(ctx, n, max_len, seed, corrupt):
    """schemes randomly interleaved; the messages of the Ed25519 items in order (the others have none)"""
    rng = np.random.default_rng(seed)
    counts = [int(round(n * MIX[0])), int(round(n * MIX[1]))]
    counts.append(n - sum(counts))
    schemes = np.repeat(np.arange(3, dtype=np.uint8), counts)
    rng.shuffle(schemes)
    lens = np.zeros(n, np.int64)
    lens[schemes == 2] = _lengths(rng, counts[2], max_len, True)
    d_schemes = torch.from_numpy(schemes).cuda()
    sigs, aux = _bytes(n, 64), _bytes(n, 32)
    for curve in (0, 1):
        at = d_schemes == curve
        if counts[curve]:
            s, d, _ = _gen_secp(ctx, curve, counts[curve], 3 * seed + curve, corrupt)
            sigs[at], aux[at] = s, d
    s, k, msgs, _ = _gen_ed25519(ctx, lens[schemes == 2], 3 * seed + 2, corrupt)
    at = d_schemes == 2
    sigs[at], aux[at] = s, k
    return d_schemes, sigs, aux, msgs, torch.from_numpy(_offsets(lens)).cuda()


def _host(*tensors):
    return tuple(t.cpu().numpy() for t in tensors)


def _message_inputs(case, seed):
    """the ``digests`` kind's data: random bytes of log-uniform lengths, and their offsets"""
    off = _offsets(_lengths(np.random.default_rng(seed), case["n"], case["max_len"], True))
    g = torch.Generator(device="cuda").manual_seed(seed)
    data = torch.randint(0, 256, ((int(off[-1]) + 31) // 16 * 16,), dtype=torch.uint8, device="cuda", generator=g)
    return data, off


_servers = {}


def _server():
    # one server per process, as a service keeps it
    if "slots" not in _servers:
        _servers["slots"] = sigops.Server()
    return _servers["slots"]


def prepare(case, seed):
    ctx = sigops.default_context()
    kind, n = case["kind"], case["n"]
    device = case.get("where") == "device"
    state = dict(case=case, ctx=ctx)
    if kind in ("recover", "address", "verify"):
        sigs, digests, keys = _gen_secp(ctx, case["curve"], n, seed, case["corrupt"])
        ins = (sigs, digests, keys) if kind == "verify" else (sigs, digests)
        state["ins"] = ins if device else _host(*ins)
        state["out"] = (_bytes(n, 64), _bytes(n, 0))
    elif kind in ("ed25519", "ed25519_strict"):
        lens = _lengths(np.random.default_rng(seed), n, case["max_len"], case["log_lengths"])
        ins = _gen_ed25519(ctx, lens, seed, case["corrupt"])
        state["ins"] = ins if device else _host(*ins)
        state["out"] = (_bytes(n, 0),)
    elif kind == "mixed":
        ins = _gen_mixed(ctx, n, case["max_len"], seed, case["corrupt"])
        state["ins"] = ins if device else _host(*ins)
        state["out"] = (_bytes(n, 64), _bytes(n, 0))
    elif kind == "digests":
        data, off = _message_inputs(case, seed)
        state["ins"] = (data, torch.from_numpy(off).cuda())
        state["out"] = (_bytes(n, 32),)
    else:
        state["server"] = _server()
        # sizes log-uniform over 1..4096, the same ones for every seed, in an order of the seed's
        sizes = np.floor(4096.0 ** ((np.arange(n) + 0.5) / n)).astype(np.int64)
        req = _offsets(np.random.default_rng(seed).permutation(sizes))
        schemes, sigs, aux, msgs, off = _host(*_gen_mixed(ctx, int(req[-1]), case["max_len"], seed, case["corrupt"]))
        state["requests"] = [
            (schemes[a:b], sigs[a:b], aux[a:b], msgs[off[a]:off[b]], (off[a:b + 1] - off[a]).astype(np.uint64))
            for a, b in zip(req[:-1], req[1:])]
    return state


# ---- one pass ----

def run(state):
    case, ctx = state["case"], state["ctx"]
    kind, n = case["kind"], case["n"]
    if kind == "serve":
        server = state["server"]
        tickets = [server.submit(*request) for request in state["requests"]]
        done = [server.wait(t) for t in tickets]
        return [np.concatenate([d[0] for d in done]), np.concatenate([d[1] for d in done])]
    if case["where"] == "host":
        if kind == "recover":
            return (ctx.secp256k1_recover if case["curve"] == 0 else ctx.secp256r1_recover)(*state["ins"])
        if kind == "address":
            return ctx.recover_address(case["curve"], *state["ins"])
        if kind == "verify":
            return (ctx.secp256k1_verify if case["curve"] == 0 else ctx.secp256r1_verify)(*state["ins"])
        if kind == "mixed":
            return ctx.batch(*state["ins"])
        return ctx.ed25519_verify(*state["ins"], strict=kind == "ed25519_strict")
    ins = [t.data_ptr() for t in state["ins"]]
    out = [t.data_ptr() for t in state["out"]]
    s = _stream()
    if kind == "recover":
        ctx.secp_recover_dev(case["curve"], *ins, n, *out, s)
    elif kind == "verify":
        (ctx.secp256k1_verify_dev if case["curve"] == 0 else ctx.secp256r1_verify_dev)(*ins, n, out[1], s)
        return state["out"][1]
    elif kind == "ed25519":
        ctx.ed25519_verify_dev(*ins, n, *out, s)
    elif kind == "ed25519_strict":
        ctx.ed25519_verify_strict_dev(*ins, n, *out, s)
    elif kind == "mixed":
        ctx.batch_dev(*ins, n, *out, s)
    else:
        ctx.message_new_dev(*ins, n, *out, s)
    return list(state["out"])


# ---- what a pass cannot do without ----

# field products per item: the square roots, one doubling chain (halved by the endomorphism or the
# lattice), one addition per 4-bit window of the variable point and per 16 bits of the fixed one
PRODUCTS = {0: 269 + 128 * 7 + 64 * 11 + 16 * 11, 1: 260 + 252 * 8 + 63 * 11 + 16 * 11,
            2: 2 * 264 + 136 * 7 + 68 * 8 + 16 * 7}
PRODUCT_OPS = 2 * 64  # one 256-bit product: 64 multiply-adds of 32-bit words
SHA512_OPS = 80 * 60  # 64-bit operations per 128-byte block
SHA256_OPS = 64 * 40  # 32-bit operations per 64-byte block


def work(case):
    kind, n = case["kind"], case["n"]
    mean = 0.0
    if case.get("max_len"):
        m = case["max_len"]
        mean = m / 2 if case.get("log_lengths") is False else m / np.log(m + 1)
    ed = dict(bytes=64 + 32 + 8 + mean + 1, flops=PRODUCTS[2] * PRODUCT_OPS + (mean + 81) / 128 * SHA512_OPS)
    if kind in ("recover", "address", "verify"):
        per = dict(bytes=96 + {"recover": 65, "address": 33, "verify": 65}[kind],
                   flops=(PRODUCTS[case["curve"]] - (269 if kind == "verify" else 0)) * PRODUCT_OPS)
    elif kind in ("ed25519", "ed25519_strict"):
        per = ed
    elif kind == "digests":
        per = dict(bytes=mean + 8 + 32, flops=(mean + 73) / 64 * SHA256_OPS)
    else:
        per = dict(bytes=97 + 8 + 65 + MIX[2] * mean,
                   flops=MIX[0] * PRODUCTS[0] * PRODUCT_OPS + MIX[1] * PRODUCTS[1] * PRODUCT_OPS + MIX[2] * ed["flops"])
        if kind == "serve":
            n = n * 4095 / np.log(4096.0)  # the mean request
    return {"bytes": float(per["bytes"] * n), "flops": float(per["flops"] * n)}


def exact(case, seed):
    """digests by hashlib; the other inputs are signed by the library's own generator, so their keys
    and statuses have no value made without it"""
    if case["kind"] != "digests":
        return None
    data, off = _message_inputs(case, seed)
    raw = data.cpu().numpy().tobytes()
    out = b"".join(hashlib.sha256(raw[a:b]).digest() for a, b in zip(off[:-1], off[1:]))
    return [torch.from_numpy(np.frombuffer(out, np.uint8).reshape(-1, 32).copy())]
