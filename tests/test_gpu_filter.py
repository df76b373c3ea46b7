"""GPU test of the filter pipeline, which serves large k in the library's own configuration: a sampled
bound, one pass over the keys, selection of what it keeps.  Outputs must equal the oracle's and the
general pipeline's (the same call with stats) bit for bit: every sample size, ragged ends, keys that
tie at and above the bound, clustered keys that leave their unit's segment, and keys planted to
defeat the sample."""
import numpy as np
import pytest

from test_gpu_short import check, dt, make  # noqa: F401

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# (n, k): the sample is 2^13 from k = n/256, 2^15, 2^17, 2^19 below; k = n/8 and n/4; ragged ends
CASES = [(36865, 4608), (65537, 16384), (73_737, 9_217), (131_073, 9000), (1_000_003, 9_001), ((1 << 20) + 7, 131_072),
         ((1 << 24) + 5, 1 << 16), ((1 << 24) - 1, 9_000), (1 << 24, 1 << 22), (1 << 25, 8_300), (40_000_003, 9_000),
         (50_000_001, 365_353), ((1 << 26) + 1, 300_000), ((1 << 27) + 3, (1 << 23) + 70_001)]


@pytest.mark.parametrize("n,k", CASES)
@pytest.mark.parametrize("dist", ["uniform", "f32"])
def test_large_k(orc, dt, dist, n, k):  # noqa: F811
    v, f32 = make(orc, dist, n, 29)
    print(f"[case] filter {dist} n={n} k={k}", flush=True)
    check(orc, dt, v, f32, k, dt.ALGO_RADIX)
    if n < 1 << 20:
        check(orc, dt, v, f32, k, dt.ALGO_RADIX, alpha=-2)
        check(orc, dt, v, f32, k, dt.ALGO_BUCKET)


@pytest.mark.parametrize("dist", ["lognormal", "equal", "zeros", "few", "ascending", "descending", "f32_special",
                                  "steps", "tail", "block"])
@pytest.mark.parametrize("n,k", [(131_075, 16_000), ((1 << 20) + 3, 20_000), ((1 << 24) + 1, 1 << 17)])
def test_large_k_tied_and_clustered(orc, dt, dist, n, k):  # noqa: F811
    rng = np.random.default_rng(31)
    f32 = False
    if dist == "steps":  # a thousand values, each many times, far apart
        v = (rng.integers(0, 1000, n) * 4_000_000).astype(np.uint32)
    elif dist == "tail":  # heavy tail: most of the range above the bound is empty
        v = np.minimum(2.0 ** 32 - 1, 1000.0 / (1.0 - rng.random(n))).astype(np.uint32)
    elif dist == "block":  # one run of large keys
        v = rng.integers(0, 1 << 20, n, dtype=np.uint32)
        v[n // 3:n // 3 + n // 16] += np.uint32(1 << 21)
    else:
        v, f32 = make(orc, dist, n, 37)
    print(f"[case] filter {dist} n={n} k={k}", flush=True)
    check(orc, dt, v, f32, k, dt.ALGO_RADIX)


def sample_positions(n, lm):
    """Positions of the sampled keys: one per stratum [i n / m, (i + 1) n / m)."""
    i = np.arange(1 << lm, dtype=np.uint64)
    b, e = (i * np.uint64(n)) >> np.uint64(lm), ((i + np.uint64(1)) * np.uint64(n)) >> np.uint64(lm)
    h = (i.astype(np.uint32) * np.uint32(0x9E3779B1)).astype(np.uint32)
    for s, m in ((15, 0x85EBCA77), (13, 0xC2B2AE3D), (16, None)):
        h = h ^ (h >> np.uint32(s))
        if m is not None:
            h = (h * np.uint32(m)).astype(np.uint32)
    return (b + ((h.astype(np.uint64) * (e - b)) >> np.uint64(32))).astype(np.int64)


@pytest.mark.parametrize("n,k,lm", [(1_000_001, 20_000, 13), (2_400_003, 9_000, 15), ((1 << 24) + 1, 9_000, 17)])
@pytest.mark.parametrize("planted", ["high", "low"])
def test_sample_defeated(orc, dt, planted, n, k, lm):  # noqa: F811
    """The sampled keys are the largest (the bound lets too few keys through) or the smallest of all
    (it lets nearly every key through): the exact selection takes over."""
    v, _ = make(orc, "uniform", n, 41)
    v = (v >> np.uint32(1)) + np.uint32(1 << 30)
    pos = sample_positions(n, lm)
    rng = np.random.default_rng(5)
    v[pos] = rng.integers(0, 1 << 29, pos.size, dtype=np.uint32) + np.uint32((1 << 32) - (1 << 29) if planted == "high" else 0)
    print(f"[case] filter sample {planted} n={n} k={k}", flush=True)
    check(orc, dt, v, False, k, dt.ALGO_RADIX)


def test_large_k_partial_outputs_and_graph(orc, dt):  # noqa: F811
    n, k = 1_000_003, 30_000
    vs = [make(orc, "uniform", n, s)[0] for s in (1, 2)]
    dev = torch.from_numpy(vs[0].view(np.int32)).cuda()
    K, keys, idx = orc.topk_reference(vs[0], k)
    print("[case] filter partial outputs", flush=True)
    kth, _, _, _ = dt.select(dev, k, want_keys=False, want_idx=False)
    _, tk, _, _ = dt.select(dev, k, want_idx=False)
    _, _, ti, _ = dt.select(dev, k, want_keys=False)
    torch.cuda.synchronize()
    assert int(kth.cpu().numpy().view(np.uint32)[0]) == K
    assert np.array_equal(tk.cpu().numpy().view(np.uint32), keys) and np.array_equal(ti.cpu().numpy(), idx)
    ws = torch.empty(dt.workspace_size(n, k), dtype=torch.uint8, device="cuda")
    out = (torch.empty(1, dtype=torch.int32, device="cuda"), torch.empty(k, dtype=torch.int32, device="cuda"),
           torch.empty(k, dtype=torch.int64, device="cuda"))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        dt.select(dev, k, workspace=ws, out=out)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    print("[case] filter graph", flush=True)
    with torch.cuda.graph(g, stream=s):
        dt.select(dev, k, workspace=ws, out=out, stream=torch.cuda.current_stream())
    for v in vs * 2:
        dev.copy_(torch.from_numpy(v.view(np.int32)))
        g.replay()
        torch.cuda.synchronize()
        K, keys, idx = orc.topk_reference(v, k)
        assert int(out[0].cpu().numpy().view(np.uint32)[0]) == K
        assert np.array_equal(out[1].cpu().numpy().view(np.uint32), keys)
        assert np.array_equal(out[2].cpu().numpy(), idx)


@pytest.mark.parametrize("n,k", [((1 << 26) + 3, 70_000), (1 << 26, (1 << 21) + 1)])
@pytest.mark.parametrize("dist", ["ascending", "block", "runs"])
def test_dense_units(orc, dt, dist, n, k):  # noqa: F811
    """Kept keys that fill their units: sorted keys, one block of large ones, long runs of equal ones."""
    if dist == "block":
        v = make(orc, "uniform", n, 47)[0] >> np.uint32(4)
        v[n // 5:n // 5 + k + 1000] |= np.uint32(1 << 31)
    elif dist == "runs":
        v = (np.arange(n, dtype=np.uint64) // 5000 * 2654435761 % (1 << 32)).astype(np.uint32)
    else:
        v = make(orc, "ascending", n, 47)[0]
    print(f"[case] filter dense {dist} n={n} k={k}", flush=True)
    check(orc, dt, v, False, k, dt.ALGO_RADIX)


def test_longest_ranges(orc, dt):  # noqa: F811
    """2^29 keys with few kept: ranges of as many units as one holds; the same call with stats takes the
    general pipeline."""
    n, k = 1 << 29, 40_000
    x = torch.randint(-(1 << 31), (1 << 31) - 1, (n,), device="cuda", dtype=torch.int32)
    print("[case] filter 2^29", flush=True)
    a = dt.select(x, k)
    b = dt.select(x, k, stats=True)
    torch.cuda.synchronize()
    for p, q in zip(a[:3], b[:3]):
        assert torch.equal(p, q)
