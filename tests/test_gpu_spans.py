"""New mutations in spans (gf_const_drift.hpp: drift_span): launches with
enough births for one and for two tiles a wave, of a length that is and is not
a multiple of a Philox block, with samples and preserved mutations, against the
CPU oracle, and batches whose layout takes them against single runs, bit for
bit."""
import numpy as np
import pytest

from parallelpopgen_amd import scenarios as S
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu


# 6e4 births a generation: from 5 generations on (3.0e5) a tile a wave, from
# 35 (2.1e6) two
@pytest.mark.parametrize("kpl", [0, 5, 6, 35, 40])
@pytest.mark.parametrize("s,h,preserve,sample", [(0.0, 0.5, 0, 0), (-0.01, 0.0, 11, 23)])
def test_spans_against_oracle(gpu, oracle, kpl, s, h, preserve, sample):
    d = S.constant(N=1000, L=3e10, G=41, s=s, h=h, compact_interval=9, preserve_every=preserve, sample_every=sample)
    gpu.set_generations_per_launch(kpl)
    try:
        a = gpu.run(d)
    finally:
        gpu.set_generations_per_launch(0)
    assert_same(a, oracle.run(d), (kpl, s))


# a layout of more than 65,536 tiles: 76 simulations of 2e4 births a
# generation (280,000 slots and more each), 12 of 2 to 500, which stay below a
# group of tiles of new mutations
@pytest.mark.parametrize("K", [5, 8, 32])
def test_batch_spans(gpu, K):
    n = 88
    rng = np.random.default_rng(K)
    sims = np.zeros(n, gpu.BATCH_SIM_DTYPE)
    sims["N"] = rng.integers(60, 2000, n)
    sims["N1"] = np.where(rng.random(n) < 0.3, sims["N"] * 3, 0)
    sims["F"] = rng.uniform(0, 0.2, n)
    sims["h"] = 0.3
    sims["s"] = rng.uniform(-0.02, 0.002, n)
    sims["mu"] = 1e-8
    births = np.where(np.arange(n) % 8 < 7, 2e4, np.exp(rng.uniform(np.log(2), np.log(500), n)))
    sims["num_sites"] = births / (2e-8 * sims["N"])
    sims["num_generations"] = rng.integers(1, 90, n)
    sims["seed1"], sims["seed2"] = np.arange(n) + 3, 7
    gpu.set_generations_per_launch(K)
    try:
        b = gpu.batch_run(sims, compact_interval=16, sfs_n=30, keep_states=True)
    finally:
        gpu.set_generations_per_launch(0)
    live = 0
    for k in range(n):
        a = gpu.run(S.sweep_plain_desc(sims[k], 16))
        last = a["samples"][-1]
        f, ids = b["states"][k]
        assert np.array_equal(last["freq"][0].view(np.uint32), f.view(np.uint32)), k
        assert np.array_equal(a["ids"], ids), k
        live += int(a["live"][1:].sum())
    assert live == b["live_mutation_generations"]


# the tile scan's two forms: around one chunk (4,096 tiles), several, and the
# last count that a workgroup adds up itself (65,536)
@pytest.mark.parametrize("L", [3.1e10, 3.4e10, 1.6e11, 5.5e11])
def test_tile_scan_sizes(gpu, oracle, L):
    d = S.constant(N=1000, L=L, G=3, s=-0.001, compact_interval=1)
    gpu.set_generations_per_launch(1)
    try:
        a = gpu.run(d)
    finally:
        gpu.set_generations_per_launch(0)
    assert_same(a, oracle.run(d), L)
