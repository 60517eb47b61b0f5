"""The count form of the single-population drift (gf_const_drift.hpp): its
draw table on the host against binom_draw, and the launches that switch into
and out of it against the CPU oracle, bit for bit."""
import numpy as np
import pytest

from parallelpopgen_amd import scenarios as S
from parallelpopgen_amd.capi import BATCH_SIM_DTYPE, GF_INIT_PREV
from test_gpu_parity import assert_same
from test_host_math import run_host_check


def test_draw_table_equals_the_inversion():
    assert "every lookup equals binom_draw" in run_host_check("pois_rows")


# chromosome numbers at the edges of the count form's range (100 .. 2^21), with
# counts whose mean stays in the table far past 6 (s = -0.5) or leaves it early
@pytest.mark.gpu
@pytest.mark.parametrize("N,s,h,L", [(49, 0.0, 0.5, 3e9), (50, 0.02, 1.0, 3e9), (51, -0.5, 0.5, 3e9),
                                     (64, -1.0, 1.0, 3e9), (1 << 20, -2e-5, 0.0, 2e5), ((1 << 20) + 1, 1e-5, 0.5, 2e5)])
def test_range_edges(gpu, oracle, N, s, h, L):
    d = S.constant(N=N, L=L, G=70, s=s, h=h, F=0.0, compact_interval=9)
    assert_same(gpu.run(d), oracle.run(d), (N, s))


# size and selection change inside and at the edges of launches; launches
# shorter than a Philox block; no compaction, preserved mutations, samples
@pytest.mark.gpu
@pytest.mark.parametrize("kpl", [0, 3, 10])
@pytest.mark.parametrize("interval,preserve", [(0, 0), (13, 20)])
def test_model_changes(gpu, oracle, kpl, interval, preserve):
    d = S.constant(N=1000, L=3e8, G=96, s=-0.003, h=0.3, F=0.1, compact_interval=interval, preserve_every=preserve,
                   sample_every=31)
    p = d.params
    p["N"][1:] = 3000             # the start is counted in other chromosomes
    p["N"][40:55] = 45            # below the range
    p["sel_intercept"][60:] = 0.0
    p["sel_slope"][75:] = 0.01    # s(x), not constant
    gpu.set_generations_per_launch(kpl)
    try:
        a = gpu.run(d)
    finally:
        gpu.set_generations_per_launch(0)
    assert_same(a, oracle.run(d), (kpl, interval))


# a previous run's frequencies need not be counts of any chromosome number
@pytest.mark.gpu
def test_continuation_from_given_frequencies(gpu, oracle):
    n = 700
    rng = np.random.default_rng(3)
    f = rng.uniform(0, 1, (1, n)).astype(np.float32)
    f[0, :5] = [0.0, 1.0, 1e-30, 0.99999994, 0.5]
    ids = np.zeros(n, gpu.MUTID_DTYPE)
    ids["origin_threadID"] = np.arange(1, n + 1)
    d = S.constant(N=800, L=1e8, G=30, s=0.001, init_mode=GF_INIT_PREV, start_generation=7, init_freq=f, init_ids=ids,
                   init_extinct=np.zeros(1, np.uint8))
    assert_same(gpu.run(d), oracle.run(d), "prev")


# one batch with simulations inside and outside the range, resized or not
@pytest.mark.gpu
def test_mixed_batch(gpu):
    sims = np.zeros(12, BATCH_SIM_DTYPE)
    sims["N"] = [30, 49, 50, 500, 500, 2000, 60, 1000, 1 << 20, (1 << 20) + 1, 3000, 700]
    sims["N1"] = [0, 0, 400, 40, 500, 9000, 0, 1 << 20, 0, 0, 10, 0]
    sims["F"], sims["h"], sims["mu"] = 0.0, 0.5, 1e-9
    sims["s"] = [0.0, 0.01, -0.5, 0.002, -0.01, 0.0, -1.0, -0.001, 1e-5, 0.0, 0.01, -0.2]
    sims["num_sites"] = [3e9, 3e9, 1e9, 1e8, 1e8, 1e7, 1e9, 1e6, 1e5, 1e5, 1e7, 1e8]
    sims["seed1"], sims["seed2"] = 100 + np.arange(12), 5
    sims["num_generations"] = [50, 3, 41, 30, 64, 33, 20, 25, 17, 18, 40, 1]
    r = gpu.batch_run(sims, compact_interval=11, sfs_n=20, keep_states=True)
    for i, b in enumerate(sims):
        p = gpu.run(S.sweep_plain_desc(b))["samples"][-1]
        f, _ = r["states"][i]
        assert np.array_equal(f.view(np.uint32), p["freq"][0].view(np.uint32)), i


# launches whose tiles keep a handful of slots each: a wave gathers over many
# input tiles, empty ones among them (one population and two)
@pytest.mark.gpu
@pytest.mark.parametrize("P,s,kpl", [(1, -0.9, 64), (1, -0.4, 33), (2, -0.9, 48)])
def test_gather_over_sparse_tiles(gpu, oracle, P, s, kpl):
    d = S.constant(N=500, L=2e9 / P, G=140, s=s, h=0.9, P=P, m=0.01, compact_interval=kpl)
    gpu.set_generations_per_launch(kpl)
    try:
        a = gpu.run(d)
    finally:
        gpu.set_generations_per_launch(0)
    assert_same(a, oracle.run(d), (P, s, kpl))
