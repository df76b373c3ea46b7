"""GPU test of the one- and four-launch pipelines that serve calls in the library's own configuration
(automatic alpha, default options, no stats): k-th key, top-k keys and indices must equal, bit for
bit, those of the general pipeline (the same call with stats) and the oracle's, at the edges of
every register block, both levels of the first top-k and the streamed second top-k."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dt():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import drtopksc_amd as dt
    dt.lib()
    return dt


def make(orc, dist, n, seed):
    """uint32 bit patterns (and whether they are float32 keys)."""
    rng = np.random.default_rng(seed)
    if dist == "uniform":
        return orc.generate(orc.UNIFORM_U32, seed, n), False
    if dist == "lognormal":
        return orc.generate(orc.LOGNORMAL_U32, seed, n), False
    if dist == "equal":
        return np.full(n, 0x12345678, np.uint32), False
    if dist == "zeros":
        return np.zeros(n, np.uint32), False
    if dist == "few":  # zeros, the largest key and values between, heavily tied
        return rng.choice(np.array([0, 0, 1, 7, 2 ** 31, 2 ** 32 - 2, 2 ** 32 - 1], np.uint32), n), False
    if dist == "ascending":
        return np.arange(n, dtype=np.uint32) * np.uint32(3), False
    if dist == "descending":
        return (np.uint32(2 ** 32 - 1) - np.arange(n, dtype=np.uint32)), False
    if dist == "f32":
        return orc.generate(orc.NORMAL_F32, seed, n), True
    assert dist == "f32_special"  # infinities, NaN of both signs, both zeros among ordinary keys
    v = rng.standard_normal(n).astype(np.float32).view(np.uint32)
    sp = np.array([0x7F800000, 0xFF800000, 0x7FC00000, 0xFFC00000, 0x00000000, 0x80000000, 0x7F7FFFFF], np.uint32)
    at = rng.integers(0, n, max(1, n // 8))
    v[at] = sp[rng.integers(0, sp.size, at.size)]
    return v, True


def check(orc, dt, v, f32, k, algo, alpha=-1):
    dev = torch.from_numpy(v.view(np.float32 if f32 else np.int32)).cuda()
    o = orc.f32_to_ordered(v) if f32 else v
    K, keys, idx = orc.topk_reference(o, k)
    p = dt.params(alpha=alpha)
    ws = torch.full((dt.workspace_size(v.size, k, algo, 1 if f32 else 0, p),), 0xA5, dtype=torch.uint8, device="cuda")
    for rep in range(2):  # the second call meets the first one's scratch
        kth, tk, ti, _ = dt.select(dev, k, algo=algo, p=p, workspace=ws)
        torch.cuda.synchronize()
        got = [x.cpu().numpy().view(np.uint32) for x in (kth, tk)]
        if f32:
            got = [orc.f32_to_ordered(x) for x in got]
        assert int(got[0][0]) == K
        assert np.array_equal(ti.cpu().numpy(), idx)
        assert np.array_equal(got[1], keys)
    assert dt.workspace_check(ws) == 0
    kth2, tk2, ti2, _ = dt.select(dev, k, algo=algo, p=p, stats=True, workspace=ws)
    assert torch.equal(kth.view(torch.int32), kth2.view(torch.int32))
    assert torch.equal(tk.view(torch.int32), tk2.view(torch.int32)) and torch.equal(ti, ti2)


SMALL = [(1, 1), (2, 2), (3, 1), (4, 3), (5, 5), (63, 7), (255, 255), (257, 100), (4095, 10), (4096, 4096), (4097, 1),
         (8192, 300), (12289, 8000), (20_000, 1), (36863, 36863), (36864, 20000)]


@pytest.mark.parametrize("dist", ["uniform", "lognormal", "equal", "zeros", "few", "ascending", "descending", "f32",
                                  "f32_special"])
def test_one_workgroup(orc, dt, dist):
    for n, k in SMALL:
        v, f32 = make(orc, dist, n, n + 3)
        print(f"[case] small {dist} n={n} k={k}", flush=True)
        check(orc, dt, v, f32, k, dt.ALGO_RADIX)
    check(orc, dt, v, f32, 64, dt.ALGO_BUCKET)


# n above the one-workgroup limit: one, two and three levels of delegates, ragged ends, the largest
# k and k above it
SHORT = [(36865, 1), (36865, 4608), (65537, 8192), (100_003, 9000), (200_001, 25), (1_000_003, 100),
         ((1 << 20) + 1, 8192), (1 << 22, 4096), ((1 << 24) + 5, 8192), ((1 << 24) - 3, 3000), ((1 << 25) + 2, 1000),
         ((1 << 26) + 7, 8192), ((1 << 26) + 5, 16)]


@pytest.mark.parametrize("n,k", SHORT)
@pytest.mark.parametrize("dist", ["uniform", "f32"])
def test_few_launches(orc, dt, dist, n, k):
    v, f32 = make(orc, dist, n, 17)
    print(f"[case] short {dist} n={n} k={k}", flush=True)
    check(orc, dt, v, f32, k, dt.ALGO_RADIX)
    if n < 1 << 22:
        check(orc, dt, v, f32, k, dt.ALGO_RADIX, alpha=-2)
        check(orc, dt, v, f32, k, dt.ALGO_BUCKET)


# tied and clustered keys fill the concatenation up to whole subranges: the streamed second top-k
@pytest.mark.parametrize("dist", ["lognormal", "equal", "zeros", "few", "ascending", "descending", "f32_special"])
@pytest.mark.parametrize("n,k", [(65539, 777), ((1 << 20) + 3, 5000), ((1 << 22) + 1, 8192), ((1 << 25) + 9, 1024)])
def test_few_launches_clustered(orc, dt, dist, n, k):
    v, f32 = make(orc, dist, n, 23)
    print(f"[case] short {dist} n={n} k={k}", flush=True)
    check(orc, dt, v, f32, k, dt.ALGO_RADIX)


def test_outputs_may_be_left_out(orc, dt):
    for n in (3001, 300_000):
        v, _ = make(orc, "uniform", n, 5)
        dev = torch.from_numpy(v.view(np.int32)).cuda()
        K, keys, idx = orc.topk_reference(v, 50)
        print(f"[case] partial outputs n={n}", flush=True)
        kth, _, _, _ = dt.select(dev, 50, want_keys=False, want_idx=False)
        _, tk, _, _ = dt.select(dev, 50, want_idx=False)
        _, _, ti, _ = dt.select(dev, 50, want_keys=False)
        torch.cuda.synchronize()
        assert int(kth.cpu().numpy().view(np.uint32)[0]) == K
        assert np.array_equal(tk.cpu().numpy().view(np.uint32), keys) and np.array_equal(ti.cpu().numpy(), idx)


def test_graph_replay(orc, dt):
    """Captured small and four-launch calls, replayed on new keys in the same buffers."""
    for n, k in ((3001, 10), (1_000_003, 100)):
        vs = [make(orc, "uniform", n, s)[0] for s in (1, 2, 3)]
        dev = torch.from_numpy(vs[0].view(np.int32)).cuda()
        ws = torch.empty(dt.workspace_size(n, k), dtype=torch.uint8, device="cuda")
        out = (torch.empty(1, dtype=torch.int32, device="cuda"), torch.empty(k, dtype=torch.int32, device="cuda"),
               torch.empty(k, dtype=torch.int64, device="cuda"))
        print(f"[case] graph n={n} k={k}", flush=True)
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
