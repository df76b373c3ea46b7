"""GPU test of the short pipeline's second top-k on inputs that single out one branch of it each: sparse
keys, whose k-th key lies in the bucket that starts at the lowest key of all, ties that fill the k-th key's
bucket of a concatenation held in LDS, concatenations that LDS does not hold, reduced by one workgroup or
several, with every way to go on from there, and one value that most keys share.  Outputs must equal the
oracle's and the general pipeline's (the same call with stats) bit for bit."""
import numpy as np
import pytest

from test_gpu_short import check, dt  # noqa: F401

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def as_keys(orc, ordered, f32):
    """The key bits of ordered values."""
    if not f32:
        return ordered
    return np.where(ordered >> 31 != 0, ordered ^ np.uint32(1 << 31), ~ordered).astype(np.uint32)


@pytest.mark.parametrize("alpha", [-1, -2])
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,k", [(65_537, 9), (70_000, 12), (100_003, 17), (131_073, 5), (140_000, 5), (200_001, 8),
                                 (262_147, 33), (300_001, 2), (600_000, 20), (1 << 20, 64), ((1 << 20) + 3, 8)])
def test_sparse_keys(orc, dt, alpha, f32, n, k):  # noqa: F811
    """The lowest key everywhere but in 1 .. k-1 subranges of 32, one key far above the rest: the threshold
    is the lowest key, and so is the start of the k-th key's bucket."""
    rng = np.random.default_rng(n + k)
    for live in sorted({1, k // 2, k - 1} - {0}):
        v = np.zeros(n, np.uint32)
        for i, s in enumerate(rng.choice(n // 32, live, replace=False)):
            v[32 * s:32 * s + 32] = np.arange(32) if i else np.concatenate(([1 << 31], np.arange(1, 32)))
        print(f"[case] sparse n={n} k={k} alpha={alpha} f32={f32} live={live}", flush=True)
        check(orc, dt, as_keys(orc, v, f32), f32, k, dt.ALGO_RADIX, alpha=alpha)


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,k", [(100_003, 900), (1 << 20, 4000), ((1 << 22) + 1, 4096), ((1 << 22) + 5, 8192)])
def test_tied_bucket(orc, dt, f32, n, k):  # noqa: F811
    """Half of the top keys lie above one value that many neighbouring keys share: the k-th key is that value,
    far more than 256 keys are in its bucket, and the threshold lies below it."""
    for seed in range(3):
        rng = np.random.default_rng(n + seed)
        v = rng.integers(1 << 28, 1 << 30, n, dtype=np.uint32)
        top = rng.choice(n, k // 2, replace=False)
        v[top] = rng.integers(1 << 31, (1 << 32) - 1, top.size, dtype=np.uint32)
        tie = int(rng.integers(0, n - k))
        v[tie:tie + 3 * k // 4] = np.uint32((1 << 30) + 12345)
        print(f"[case] tied bucket n={n} k={k} f32={f32} seed={seed}", flush=True)
        check(orc, dt, as_keys(orc, v, f32), f32, k, dt.ALGO_RADIX)


def clustered(kind, n, k, seed):
    """Ordered keys whose k selected subranges hold far more keys >= the threshold than k."""
    rng = np.random.default_rng(seed)
    v = rng.integers(0, 1 << 20, n, dtype=np.uint32)
    lo, hi = n // 3, n // 3 + n // 16
    if kind == "scatter":  # fewer than k keys above the threshold, in as many segments
        v[:] = 0
        v[rng.integers(0, n, k // 2)] = rng.integers(1, 1 << 31, k // 2, dtype=np.uint32)
    elif kind == "ascending":
        v = np.arange(n, dtype=np.uint32) * np.uint32(5)
    elif kind == "saw":
        v = np.arange(n, dtype=np.uint32) % np.uint32(100_003)
    elif kind == "block":
        v[lo:hi] += np.uint32(1 << 21)
    elif kind == "block+outlier":  # logarithmic buckets
        v[lo:hi] += np.uint32(1 << 21)
        v[5] = np.uint32(2 ** 32 - 1)
    elif kind == "constant":  # the k-th key's bucket is one value
        v[lo:hi] = np.uint32(1 << 21)
    elif kind == "constant+above":
        v[lo:hi] = np.uint32(1 << 21)
        v[rng.integers(0, n, k // 3)] = np.uint32(3 << 20) + rng.integers(0, 1 << 19, k // 3, dtype=np.uint32)
    else:
        assert kind == "narrow"  # three values in it, each many times, and keys far above
        v[lo:hi] = np.uint32(1 << 29) + rng.integers(0, 3, hi - lo, dtype=np.uint32)
        v[rng.integers(0, n, k // 3)] = np.uint32(1 << 31) + rng.integers(0, 1 << 30, k // 3, dtype=np.uint32)
    return v


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,k", [((1 << 20) + 3, 4096), ((1 << 22) + 1, 6000), ((1 << 24) + 5, 4096)])
@pytest.mark.parametrize("kind", ["scatter", "ascending", "saw", "block", "block+outlier", "constant", "constant+above",
                                  "narrow"])
def test_long_concatenations(orc, dt, kind, n, k, f32):  # noqa: F811
    assert dt.select_route(n, k)["pipeline"] == "short"
    v = clustered(kind, n, k, n)
    print(f"[case] concatenation {kind} n={n} k={k} f32={f32}", flush=True)
    check(orc, dt, as_keys(orc, v, f32), f32, k, dt.ALGO_RADIX)


@pytest.mark.parametrize("n,k", [(257, 100), (4096, 1000), (36_864, 30_000), (300_001, 2_000)])
@pytest.mark.parametrize("share", [1.0, 0.9, 0.3])
def test_heavy_value(orc, dt, share, n, k):  # noqa: F811
    """One value that most keys share, an outlier above and a few keys below: every pass of a selection meets
    waves full of one bucket."""
    rng = np.random.default_rng(n)
    v = rng.integers(0, 1 << 31, n, dtype=np.uint32)
    v[rng.random(n) < share] = 1000
    v[n // 3] = np.uint32(2 ** 32 - 1)
    v[n // 2:n // 2 + 16] = 5
    print(f"[case] heavy value n={n} k={k} share={share}", flush=True)
    check(orc, dt, v, False, k, dt.ALGO_RADIX)


def test_long_concatenations_in_a_graph(orc, dt):  # noqa: F811
    """A captured call, replayed on keys that go through the several workgroups, through one and back: the
    arrivals are counted anew in each replay."""
    n, k = (1 << 22) + 1, 6000
    vs = [clustered(kind, n, k, 3) for kind in ("block", "ascending", "scatter", "constant")]
    dev = torch.from_numpy(vs[0].view(np.int32)).cuda()
    ws = torch.empty(dt.workspace_size(n, k), dtype=torch.uint8, device="cuda")
    out = (torch.empty(1, dtype=torch.int32, device="cuda"), torch.empty(k, dtype=torch.int32, device="cuda"),
           torch.empty(k, dtype=torch.int64, device="cuda"))
    print(f"[case] concatenation graph n={n} k={k}", flush=True)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        dt.select(dev, k, workspace=ws, out=out)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
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
