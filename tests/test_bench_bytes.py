"""bench.py's byte counts, on the CPU: a call's fraction of the HBM peak comes from the pipeline that serves it,
not from the statistics of the general one."""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def stats(n, k, alpha=4):
    """What the general pipeline reports where nearly every subrange is selected (13.8% of the keys tie at the top)."""
    S = n >> alpha
    return {"alpha": alpha, "path": 2, "num_delegates": 2 * S, "concat_size": n // 4, "selected_subranges": S,
            "first_passes": 2, "second_passes": 4, "count_greater": 0, "phase_ms": [0.0] * 5}


def route(pipeline, **kw):
    return dict({"pipeline": pipeline, "alpha": 0, "sample_log2": 0, "last_resort": 0, "delegates": 0, "slots": 0,
                 "kept": 0}, **kw)


def test_fractions_stay_below_the_peak(bench):
    n, k = 1 << 30, 1 << 22
    st = stats(n, k)
    ms = 0.7  # measured for such keys on the filter pipeline: the keys alone take 0.54 ms at the peak
    assert bench.frac(bench.bytes_general(st, n, k), ms) > 1
    r = bench.row(route("filter", kept=k), st, n, k, ms)
    assert r["hbm_frac_4n"] <= r["hbm_frac"] < 1 and "hbm_frac_survey" not in r
    assert r["stats_call"]["alpha"] == 4


def test_bytes_of_each_pipeline(bench):
    n, k = 1 << 20, 100
    st = stats(n, k)
    out = 12 * k
    assert bench.bytes_moved(route("small"), st, n, k) == 4 * n + out
    assert bench.bytes_moved(route("short", delegates=4096, slots=k << 8), st, n, k) == 4 * n + 8 * 4096 + 4 * (k << 8) + 16 * k + out
    assert bench.bytes_moved(route("filter"), dict(st, count_greater=90), n, k) == 4 * n + 20 * 90 + out
    assert bench.bytes_moved(route("general"), st, n, k) == bench.bytes_general(st, n, k)


def test_the_line_is_brief(bench):
    n, k = 1 << 30, 1 << 10
    rows = [bench.row(route("short", delegates=1 << 18, slots=k << 12), stats(n, k), n, k << j, 0.7) for j in range(25)]
    b = bench.brief({"a": {"dist": "x", "radix": rows, "few": rows[::4]}, "none": None})
    assert b["a"]["radix"] == [0.7] * 25 and b["a"]["few"][1] == [k << 4, 0.7] and b["a"]["dist"] == "x" and b["none"] is None
