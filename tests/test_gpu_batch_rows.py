"""GPU test of the batched rows selected in LDS: arrays at, one below and one above what LDS stages (14336
delegates or keys, 4096 listed subranges, 6144 concatenated keys), tied so that the concatenation is as long
as it gets, and rows of one queue that alternate between the LDS selection and the digit passes.  Outputs must
equal the oracle's bit for bit."""
import pytest

from test_gpu_batch import check, dt, make_rows, run_batch  # noqa: F401

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("alpha", [0, 1, 3, 6])
@pytest.mark.parametrize("kind", ["rand", "ties", "equal"])
def test_row_capacities(orc, dt, alpha, kind):  # noqa: F811
    specs = []
    for i, S in enumerate((1, 3, 2047, 2049, 14335, 14336, 14337)):
        n = S << alpha
        for j, k in enumerate((1, 95, 97, 4095, 4096, 4097, 6144, 6145)):
            if k <= S:
                specs.append((n - (j % 3 if n > 3 * 64 and alpha else 0), k, (i + j) & 1, kind))
    rows, buf, kl, ol, ordered = make_rows(orc, specs, seed0=3000 + alpha)
    t = dt.tuning_default()
    for d in range(2):
        for ln in range(32):
            for lk in range(32):
                t.alpha[d][ln][lk] = alpha
    print(f"[case] batch rows alpha={alpha} {kind} rows={len(rows)}", flush=True)
    b, dev, kth, tk, ti = run_batch(dt, rows, buf, kl, ol, tuning=t)
    check(orc, rows, ordered, kth, tk, ti, f"rows a{alpha} {kind}")
