"""GPU test of the filter pipeline on calls that it is known to serve (drtopk_select_route): its edges in k, a
defeated sample of every size, ties between the ranks that its splitters cover, a sample that places the k-th
key five deviations too low, and units and ranges at the edges of being full.  Outputs must equal the oracle's
and the general pipeline's bit for bit, and only a defeated sample may end in the one-workgroup selection from
all keys."""
import numpy as np
import pytest

from test_gpu_filter import sample_positions
from test_gpu_short import check, dt, make  # noqa: F401

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def filtered(dt, v, f32, k):  # noqa: F811
    """One call on the filter pipeline; whether it took the last resort."""
    dev = torch.from_numpy(v.view(np.float32 if f32 else np.int32)).cuda()
    ws = torch.empty(dt.workspace_size(v.size, k, dt.ALGO_RADIX, 1 if f32 else 0), dtype=torch.uint8, device="cuda")
    dt.select(dev, k, workspace=ws)
    r = dt.select_route(v.size, k, dtype=1 if f32 else 0, workspace=ws)
    assert r["pipeline"] == "filter"
    return r


@pytest.mark.parametrize("n,k,lm", [(65_537, 8_192, 13), (73_737, 9_217, 13), (1_000_003, 125_000, 13),
                                    ((1 << 24) + 3, 8_000, 17), ((1 << 25) + 1, 7_169, 19), (2_400_003, 8_500, 15), ((1 << 24) + 5, 1 << 22, 13), (40_000_003, 9_300, 17)])
@pytest.mark.parametrize("dist", ["uniform", "f32"])
def test_edges_in_k(orc, dt, dist, n, k, lm):  # noqa: F811
    v, f32 = make(orc, dist, n, 61)
    print(f"[case] filter edge {dist} n={n} k={k}", flush=True)
    check(orc, dt, v, f32, k, dt.ALGO_RADIX)
    r = filtered(dt, v, f32, k)
    assert r["sample_log2"] == lm and r["last_resort"] == 0


@pytest.mark.parametrize("n,k,lm", [(1_000_001, 20_000, 13), (2_400_003, 8_500, 15), (40_000_003, 9_300, 17)])
def test_defeated_sample(orc, dt, n, k, lm):  # noqa: F811
    """The sampled keys are the largest: the bound lets too few keys through."""
    v, _ = make(orc, "uniform", n, 67)
    v = (v >> np.uint32(1)) + np.uint32(1 << 30)
    pos = sample_positions(n, lm)
    v[pos] = np.random.default_rng(5).integers(0, 1 << 29, pos.size, dtype=np.uint32) + np.uint32((1 << 32) - (1 << 29))
    print(f"[case] filter defeated n={n} k={k}", flush=True)
    check(orc, dt, v, False, k, dt.ALGO_RADIX)
    r = filtered(dt, v, False, k)
    assert r["sample_log2"] == lm and r["last_resort"] == 1


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,k,tied", [(1 << 25, 1_392_508, 0.0366), (1 << 24, 696_320, 0.0366), (1 << 24, 1 << 21, 0.12),
                                      ((1 << 24) + 3, 40_000, 0.0017), (1_000_003, 20_000, 0.017)])
def test_ties_above_the_kth_key(orc, dt, f32, n, k, tied):  # noqa: F811
    """Saturated keys: so many tie at the top that the tie reaches into the ranks the splitters cover, and the
    k-th key lies below it."""
    rng = np.random.default_rng(n)
    v = rng.integers(0, 1 << 30, n, dtype=np.uint32) + np.uint32(1 << 31 if f32 else 0)
    v[rng.random(n) < tied] = np.uint32((1 << 30) + (1 << 31 if f32 else 0))
    if f32:
        v ^= np.uint32(1 << 31)  # positive floats
    print(f"[case] filter saturated n={n} k={k} f32={f32}", flush=True)
    check(orc, dt, v, f32, k, dt.ALGO_RADIX)
    assert filtered(dt, v, f32, k)["last_resort"] == 0


@pytest.mark.parametrize("dist", ["lognormal", "ascending", "descending", "f32_special", "block"])
@pytest.mark.parametrize("n,k", [((1 << 20) + 3, 20_000), ((1 << 24) + 1, 1 << 17)])
def test_no_last_resort(orc, dt, dist, n, k):  # noqa: F811
    if dist == "block":
        v, f32 = np.random.default_rng(3).integers(0, 1 << 20, n, dtype=np.uint32), False
        v[n // 3:n // 3 + n // 16] += np.uint32(1 << 21)
    else:
        v, f32 = make(orc, dist, n, 71)
    print(f"[case] filter {dist} n={n} k={k}", flush=True)
    assert filtered(dt, v, f32, k)["last_resort"] == 0


@pytest.mark.parametrize("n,k", [(1 << 24, 1 << 20), (1 << 25, 1 << 22)])
def test_unlucky_sample(orc, dt, n, k):  # noqa: F811
    """Five standard deviations too few of the sampled keys are among the top k: the splitters still cover the
    k-th key."""
    lm = 13
    assert dt.select_route(n, k)["sample_log2"] == lm
    rng = np.random.default_rng(n)
    pos = sample_positions(n, lm)
    r = k * 2 ** lm / n
    high = rng.choice(pos, int(r - 5 * r ** 0.5), replace=False)
    rest = np.ones(n, bool)
    rest[pos] = False
    others = rng.choice(np.flatnonzero(rest), k - high.size, replace=False)
    v = rng.integers(0, 1 << 31, n, dtype=np.uint32)
    v[high] |= np.uint32(1 << 31)
    v[others] |= np.uint32(1 << 31)
    print(f"[case] filter unlucky n={n} k={k}", flush=True)
    check(orc, dt, v, False, k, dt.ALGO_RADIX)
    assert filtered(dt, v, False, k)["last_resort"] == 0


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("counts", [(255, 256, 257), (2048,), (2047, 1, 0, 2048), (4, 256, 0, 512, 513, 1500)])
@pytest.mark.parametrize("values", ["distinct", "tied", "ascending"])
@pytest.mark.parametrize("n,k", [((1 << 22) + 5, 20_000), ((1 << 25) + 3, 40_001)])
def test_full_units(orc, dt, values, counts, f32, n, k):  # noqa: F811
    """1.5 k large keys, so many of them in every unit of 2048 as `counts` says in turn: units and ranges at and
    beside the counts from which they are shared out over the grid."""
    rng = np.random.default_rng(n + len(counts))
    v = rng.integers(0, 1 << 30, n, dtype=np.uint32)
    unit, left, at = n // 4096, 3 * k // 2, []
    while left > 0:
        c = min(counts[(unit - n // 4096) % len(counts)], left)
        at.append(2048 * unit + np.sort(rng.choice(2048, c, replace=False)))
        unit, left = unit + 1, left - c
    at = np.concatenate(at)
    if values == "distinct":
        v[at] = rng.integers(1 << 31, 1 << 32, at.size, dtype=np.uint32)
    elif values == "tied":
        v[at] = rng.integers(0, 7, at.size, dtype=np.uint32) * np.uint32(1000) + np.uint32(1 << 31)
    else:
        v[at] = np.arange(at.size, dtype=np.uint32) + np.uint32(1 << 31)
    if f32:
        v = np.where(v >> 31 != 0, v ^ np.uint32(1 << 31), ~v).astype(np.uint32)
    print(f"[case] filter units {values} {counts} n={n} k={k} f32={f32}", flush=True)
    check(orc, dt, v, f32, k, dt.ALGO_RADIX)
    assert filtered(dt, v, f32, k)["last_resort"] == 0
