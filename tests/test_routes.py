"""Which pipeline serves a call without stats (drtopk_select_route), on the CPU: the dispatch of the short and
filter pipelines, and the sizes that other tests rely on."""
import ctypes
import os

import pytest


@pytest.fixture(scope="module")
def dt():
    import drtopksc_amd as dt
    if not os.path.exists(dt.lib_path()):
        from drtopksc_amd import build
        build.build()
    dt.lib()
    return dt


ROUTES = [
    # n, k, alpha, pipeline, log2 of the samples
    (1, 1, -1, "small", 0), (36864, 36864, -1, "small", 0), (36864, 10, -2, "small", 0),
    (140_000, 5, -2, "short", 0), (262_147, 33, -1, "short", 0), (1 << 22, 4096, -1, "short", 0), (1 << 30, 1024, -1, "short", 0),
    (73_737, 9_217, -1, "filter", 13), (73_737, 9_218, -1, "general", 0),  # k = n / 8, above
    (2_400_003, 8_500, -1, "filter", 15), (2_400_003, 9_000, -1, "filter", 13),
    (1 << 24, 1 << 22, -1, "filter", 13), (1 << 24, (1 << 22) + 1, -1, "general", 0),  # k = n / 4, above
    (40_000_003, 9_000, -1, "filter", 19), (40_000_003, 9_300, -1, "filter", 17), (1 << 28, 1 << 16, -1, "filter", 17), (1 << 30, 1 << 16, -1, "filter", 19),
    (1 << 26, 7168, -1, "short", 0), (1 << 26, 7169, -1, "filter", 19), ((1 << 24) - 1, 8192, -1, "short", 0),
    (1 << 20, 8192, -1, "short", 0), (1 << 24, 8192, -1, "filter", 17),
    (1 << 30, 1 << 28, -1, "filter", 15), ((1 << 30) + 1, 1 << 20, -1, "general", 0),
]


@pytest.mark.parametrize("n,k,alpha,pipeline,lm", ROUTES)
def test_route(dt, n, k, alpha, pipeline, lm):
    for dtype in (dt.U32, dt.F32):
        for algo in (dt.ALGO_RADIX, dt.ALGO_BUCKET):
            if algo == dt.ALGO_BUCKET and alpha == -2:
                continue
            r = dt.select_route(n, k, algo, dtype, dt.params(alpha=alpha))
            if algo == dt.ALGO_RADIX:
                assert (r["pipeline"], r["sample_log2"]) == (pipeline, lm)
            assert r["last_resort"] == 0


def test_other_configurations_keep_the_general_pipeline(dt):
    for p in (dt.params(alpha=6), dt.params(beta=3), dt.params(digit_bits=4), dt.params(num_buckets=64), dt.params(flags=0)):
        for n, k in ((3001, 10), (1 << 22, 4096), (1 << 24, 1 << 16)):
            assert dt.select_route(n, k, p=p)["pipeline"] == "general"
    for n, k in ((3001, 8), (1 << 22, 4096), (1 << 24, 1 << 16)):
        assert dt.select_route(n, k, algo=dt.ALGO_BITONIC)["pipeline"] == "general"


def test_arguments(dt):
    for n, k in ((0, 1), (10, 0), (10, 11), (1 << 31, 1)):
        with pytest.raises(dt.DrTopKError):
            dt.select_route(n, k)
    p = dt.params()
    assert dt.lib().drtopk_select_route(0, 0, 100, 10, ctypes.byref(p), None, None, None) == 1


def test_autotuner_times_the_pipeline_it_tunes(dt):
    """Every candidate of the single-vector table, the reference policy's too, runs on the general pipeline."""
    from drtopksc_amd import autotune
    for n, k in ((1 << 16, 1), (1 << 16, 1 << 12), (1 << 20, 8), (1 << 22, 1 << 10), (1 << 24, 1 << 20), (1 << 30, 1 << 16)):
        cands = autotune.single_candidates(dt, n, k)
        assert cands[0][0] == autotune.policy_alpha(n, k) and len({c[:2] for c in cands}) == len(cands)
        for a, b, p in cands:
            try:
                r = dt.select_route(n, k, p=p)
            except dt.DrTopKError:
                continue  # fewer delegates than k: the tuner leaves it out too
            assert r["pipeline"] == "general" and r["alpha"] == a
