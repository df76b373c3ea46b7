"""Timed cases of the top-k entry points, over the sizes, key types and distributions that the
benchmark and the tests use.

A case is one call pattern on one problem:

    kind "vec"    drtopksc_amd.select on one vector: radix, bucket or bitonic family, with the
                  reference's alpha policy or the measured table; `keep` tells whether the program
                  passes a workspace and output buffers that it keeps between calls (a serving or
                  training loop) or lets the call allocate them (a script)
    kind "batch"  drtopksc_amd.Batch.run on a planned batch of uneven rows with mixed key types
    kind "serve"  a burst of requests through drtopksc_amd.Server: submit all, then wait for,
                  fetch and release each in submission order

Keys are drawn on the GPU from the seed: uint32 uniform, normal(2^31, 2^28) and lognormal(20, 2)
clamped to 32 bits (13.8% of its keys saturate at 2^32-1, so ties reach into the top-k), float32
N(0, 1) and U(-1, 1).
"""
import math

import numpy as np
import torch

import drtopksc_amd as dt
from drtopksc_amd.workloads import batch_mix, pack

ALGOS = {"radix": dt.ALGO_RADIX, "bucket": dt.ALGO_BUCKET, "bitonic": dt.ALGO_BITONIC}
ALPHAS = {"auto": dt.ALPHA_AUTO, "tuned": dt.ALPHA_TUNED}
SERVER_ARENA = 2 << 30  # bytes: every listed and drawn burst fits many times over
CHUNK = 1 << 26         # keys generated at a time


def _vec(name, algo, dist, n, k, alpha="auto", keep=True):
    return {"name": name, "kind": "vec", "algo": algo, "dist": dist, "n": n, "k": k, "alpha": alpha, "keep": keep}


def _batch(name, rows, lo, hi, kmax):
    return {"name": name, "kind": "batch", "rows": rows, "lo": lo, "hi": hi, "kmax": kmax}


def _serve(name, requests, lo, hi, kmax):
    return {"name": name, "kind": "serve", "requests": requests, "lo": lo, "hi": hi, "kmax": kmax}


def listed():
    return [
        # the smallest calls: one query's scores, a few best of them, in a loop
        _vec("vec_u32_3001_k10", "radix", "u32_uniform", 3001, 10),
        # an ordinary script call: about a million scores, ragged length, nothing kept
        _vec("vec_f32_1m_k100", "radix", "f32_normal", 1_000_003, 100, keep=False),
        # a retrieval-sized call as the server issues it, with the measured table
        _vec("vec_u32_4m_k4096_tuned", "radix", "u32_uniform", 1 << 22, 4096, alpha="tuned"),
        # heavy-tailed keys with many ties at the top, large k
        _vec("vec_lognormal_16m_k65536", "radix", "u32_lognormal", (1 << 24) + 5, 1 << 16),
        # float scores of the benchmark's 2^28 workload
        _vec("vec_f32_256m_k65536", "radix", "f32_normal", 1 << 28, 1 << 16),
        # the headline sweep at a small and at a large k
        _vec("vec_u32_1g_k1024", "radix", "u32_uniform", 1 << 30, 1 << 10),
        _vec("vec_u32_1g_k4m", "radix", "u32_uniform", 1 << 30, 1 << 22),
        # the other two selection families
        _vec("bucket_normal_64m_k4096", "bucket", "u32_normal", 1 << 26, 4096),
        _vec("bitonic_f32_64m_k1024", "bitonic", "f32_normal", 1 << 26, 1024),
        # a decoding-sized batch of equal rows, and the benchmark's batch of 4096 uneven ones
        _batch("batch_64rows_128k", 64, 17, 17, 64),
        _batch("batch_4096rows", 4096, 12, 22, 4096),
        # a burst of mixed requests at the server
        _serve("serve_96_requests", 96, 10, 22, 4096),
    ]


def _log_int(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))


def draw(rng):
    kind = rng.choice(["vec"] * 5 + ["bucket", "bitonic", "batch", "batch", "serve"])
    if kind == "vec":
        n = _log_int(rng, 1 << 10, 1 << 30)
        c = _vec("", "radix", rng.choice(["u32_uniform", "u32_normal", "u32_lognormal", "f32_normal", "f32_uniform"]), n,
                 _log_int(rng, 1, min(n // 4, 1 << 22)), rng.choice(["auto", "tuned"]), rng.random() < 0.7)
    elif kind == "bucket":
        n = _log_int(rng, 1 << 16, 1 << 28)
        c = _vec("", "bucket", rng.choice(["u32_uniform", "u32_normal", "f32_normal"]), n,
                 _log_int(rng, 1, min(n // 8, 1 << 16)))
    elif kind == "bitonic":
        n = _log_int(rng, 1 << 16, 1 << 28)
        c = _vec("", "bitonic", rng.choice(["u32_uniform", "f32_normal"]), n, 1 << rng.randint(0, 12))
        c["k"] = min(c["k"], 1 << (int(math.log2(n)) - 6))
    elif kind == "batch":
        if rng.random() < 0.5:  # equal rows
            lo = hi = rng.randint(12, 20)
            rows = _log_int(rng, 8, 256)
        else:  # rows spread over a factor of 1024
            hi = rng.randint(14, 22)
            lo = hi - 10
            rows = _log_int(rng, 16, 4096)
        c = _batch("", rows, lo, hi, _log_int(rng, 16, 4096))
    else:
        c = _serve("", _log_int(rng, 8, 128), 10, rng.randint(14, 22), _log_int(rng, 16, 4096))
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs
def _keys(dist, n, g):
    """n keys on the GPU: int32 bit patterns of uint32 keys, or float32."""
    if dist == "u32_uniform":
        return torch.randint(-2 ** 31, 2 ** 31, (n,), dtype=torch.int32, device="cuda", generator=g)
    if dist == "f32_normal":
        return torch.randn(n, device="cuda", generator=g)
    if dist == "f32_uniform":
        return torch.rand(n, device="cuda", generator=g).mul_(2).sub_(1)
    out = torch.empty(n, dtype=torch.int32, device="cuda")
    for b in range(0, n, CHUNK):
        m = min(CHUNK, n - b)
        z = torch.randn(m, dtype=torch.float64, device="cuda", generator=g)
        x = z.mul_(2.0).add_(20.0).exp_() if dist == "u32_lognormal" else z.mul_(2.0 ** 28).add_(2.0 ** 31)
        v = x.add_(0.5).floor_().clamp_(0, 2.0 ** 32 - 1).to(torch.int64)
        out[b:b + m] = torch.where(v >= 2 ** 31, v - 2 ** 32, v).to(torch.int32)
    return out


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _rows(case):
    """The rows of a batch or the requests of a burst: [(offset, n, k, out_offset, dtype)].
    Lengths and k are the case's own; the seed changes the keys."""
    count = case.get("rows") or case["requests"]
    return pack(batch_mix(seed=7, nrows=count, lo=case["lo"], hi=case["hi"], kmax=case["kmax"]))


def _store(rows, keys_len, seed):
    """One key buffer with every row: uint32 uniform or float32 N(0, 1) by the row's type."""
    g = _generator(seed)
    buf = _keys("u32_uniform", keys_len, g)
    for off, n, k, oo, d in rows:
        if d == dt.F32:
            buf[off:off + n] = _keys("f32_normal", n, g).view(torch.int32)
    return buf


class _Serving:
    """A server with the store it serves; closed with the state that holds it."""

    def __init__(self, store):
        self.srv = dt.Server(store, budget_bytes=SERVER_ARENA)

    def __del__(self):
        self.srv.close()


def prepare(case, seed):
    if case["kind"] == "vec":
        keys = _keys(case["dist"], case["n"], _generator(seed))
        s = {"kind": "vec", "keys": keys, "k": case["k"], "algo": ALGOS[case["algo"]],
             "p": dt.params(alpha=ALPHAS[case["alpha"]]), "ws": None, "out": None}
        if case["keep"]:
            code = dt.F32 if keys.dtype == torch.float32 else dt.U32
            nbytes = dt.workspace_size(case["n"], case["k"], s["algo"], code, s["p"])
            s["ws"] = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
            s["out"] = (torch.empty(1, dtype=keys.dtype, device="cuda"),
                        torch.empty(case["k"], dtype=keys.dtype, device="cuda"),
                        torch.empty(case["k"], dtype=torch.int64, device="cuda"))
        return s
    rows, keys_len, out_len = _rows(case)
    store = _store(rows, keys_len, seed)
    if case["kind"] == "batch":
        b = dt.Batch(rows, keys_len, out_len)
        return {"kind": "batch", "keys": store, "batch": b, "out": b.alloc_out()}
    torch.cuda.synchronize()  # the server reads the store on streams of its own
    return {"kind": "serve", "store": store, "serving": _Serving(store),
            "requests": [(off, n, k, d) for off, n, k, oo, d in rows]}


def run(state):
    if state["kind"] == "vec":
        kth, keys, idx, _ = dt.select(state["keys"], state["k"], algo=state["algo"], p=state["p"],
                                      workspace=state["ws"], out=state["out"])
        return kth, keys, idx
    if state["kind"] == "batch":
        return state["batch"].run(state["keys"], out=state["out"])
    srv = state["serving"].srv
    tickets = [srv.submit(*q) for q in state["requests"]]
    got = []
    for t, (off, n, k, d) in zip(tickets, state["requests"]):
        got.append(srv.fetch(srv.wait(t), k))
        srv.release(t)
    return (np.array([kth for kth, _, _ in got], np.uint32), np.concatenate([top for _, top, _ in got]),
            np.concatenate([idx for _, _, idx in got]))


def work(case):
    """The keys read once; the k-th keys, top-k keys and int64 indices written once.  A key costs
    at least one comparison."""
    if case["kind"] == "vec":
        nk, ksum, calls = case["n"], case["k"], 1
    else:
        rows, _, ksum = _rows(case)
        nk, calls = sum(r[1] for r in rows), len(rows)
    return {"bytes": 4 * nk + 12 * ksum + 4 * calls, "flops": nk}


# ---------------------------------------------------------------- exact results
def _exact(bits, is_f32, k):
    """(k-th key, top-k keys, indices) of int32 bit patterns: every key above the k-th largest and
    the lowest-index keys equal to it, by ascending index."""
    u = bits.to(torch.int64) & 0xFFFFFFFF
    if is_f32:
        u = torch.where(u >= 2 ** 31, 0xFFFFFFFF - u, u + 2 ** 31)
    kth = torch.sort(u, descending=True).values[k - 1]
    above = torch.nonzero(u > kth).flatten()
    ties = torch.nonzero(u == kth).flatten()[:k - above.numel()]
    idx = torch.sort(torch.cat([above, ties])).values
    first = ties[:1]
    return bits[first], bits[idx], idx


def exact(case, seed):
    if case["kind"] == "vec":
        keys = _keys(case["dist"], case["n"], _generator(seed))
        f = keys.dtype == torch.float32
        kth, top, idx = _exact(keys.view(torch.int32), f, case["k"])
        if f:
            kth, top = kth.view(torch.float32).to(torch.float64), top.view(torch.float32).to(torch.float64)
        return kth, top, idx
    rows, keys_len, out_len = _rows(case)
    store = _store(rows, keys_len, seed)
    per_row = [_exact(store[off:off + n], d == dt.F32, k) for off, n, k, oo, d in rows]
    kth, top, idx = (torch.cat([r[i] for r in per_row]) for i in range(3))
    if case["kind"] == "batch":
        return kth, top, idx
    return kth.cpu().numpy().view(np.uint32), top.cpu().numpy().view(np.uint32), idx.cpu().numpy()
