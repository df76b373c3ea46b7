"""GPU test of the bitonic family's tiles: run lengths below eight, equal to a tile, inputs below and just above
one tile, subranges below and above the eight composites of a thread, k at the largest of the tiles.  Outputs
must equal the oracle's bit for bit."""
import pytest

from test_gpu_short import check, dt, make  # noqa: F401

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CASES = [(1, 1, -1), (3, 2, -1), (5, 4, -1), (8, 8, -1), (9, 1, -1), (2048, 2048, 0), (2049, 4, 0), (4097, 1024, 0),
         (8191, 4096, 0), (8193, 4096, 0), (30_001, 2048, 1), (30_001, 16, 2), (70_003, 512, 3), (1_000_003, 1, -1),
         (1_000_003, 1024, 5), (1_000_003, 4096, -1), ((1 << 20) + 1, 8192, -1), ((1 << 22) + 5, 128, 9)]


@pytest.mark.parametrize("n,k,alpha", CASES)
@pytest.mark.parametrize("dist", ["uniform", "f32", "few", "zeros"])
def test_tiles(orc, dt, dist, n, k, alpha):  # noqa: F811
    v, f32 = make(orc, dist, n, 43)
    print(f"[case] bitonic {dist} n={n} k={k} alpha={alpha}", flush=True)
    check(orc, dt, v, f32, k, dt.ALGO_BITONIC, alpha=alpha)
