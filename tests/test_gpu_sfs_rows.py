"""The sample spectrum at the edges of its kernels, against the CPU oracle
bit for bit: rows of 0 and 1 mutations, around one workgroup's 256, and
longer than one pass of the grid; sample sizes at and past the largest whose
sums lie in LDS (4,094); and a batch whose workgroups each finish several
simulations, some of them empty, against single runs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 101, 4094, 4095])
@pytest.mark.parametrize("M", [0, 1, 255, 257, 300001])
def test_sfs_rows(gpu, oracle, n, M):
    if n > 4000 and M > 1000:
        M = 2049
    rng = np.random.default_rng(M + n)
    f = np.exp(rng.uniform(-12, 0, M)).astype(np.float32)
    for k, v in enumerate([0.0, 1.0, 0.99999994, 1e-30][:M]):
        f[M - 1 - k] = v
    g = gpu.site_frequency_spectrum(f, n, 1e6)
    o = oracle.site_frequency_spectrum(f, n, 1e6)
    assert np.array_equal(g.view(np.uint32), o.view(np.uint32))


@pytest.mark.parametrize("S,sites", [(1, 2e4), (700, 3e3), (65, 2e6)])
def test_batch_final_spectra(gpu, S, sites):
    sims = np.zeros(S, gpu.BATCH_SIM_DTYPE)
    rng = np.random.default_rng(S)
    sims["N"] = rng.integers(20, 400, S)
    sims["h"] = 0.5
    sims["mu"] = 1e-6
    sims["num_sites"] = sites * np.exp(rng.uniform(-4, 0, S))
    sims["num_sites"][1::3] = 1.0      # most of these end with no mutation
    sims["seed1"], sims["seed2"] = np.arange(S) + 5, 9
    sims["num_generations"] = rng.integers(1, 80, S)
    n = 40
    r = gpu.batch_run(sims, sfs_n=n, keep_states=True)
    for i in range(0, S, max(1, S // 60)):
        f, _ = r["states"][i]
        one = gpu.site_frequency_spectrum(f, n, float(sims["num_sites"][i]))
        assert np.array_equal(one.view(np.uint32), r["sfs"][i].view(np.uint32))


def test_pooled_streams_and_threads(gpu, oracle):
    """more threads at once than idle streams are kept, before and after the
    pools are given back"""
    from concurrent.futures import ThreadPoolExecutor
    rng = np.random.default_rng(3)
    rows = [np.exp(rng.uniform(-9, 0, 1000 + 37 * k)).astype(np.float32) for k in range(12)]
    want = [oracle.site_frequency_spectrum(f, 60, 1e6).view(np.uint32) for f in rows]
    for _ in range(2):
        with ThreadPoolExecutor(12) as ex:
            got = list(ex.map(lambda f: gpu.site_frequency_spectrum(f, 60, 1e6).view(np.uint32), rows * 3))
        assert all(np.array_equal(g, want[k % 12]) for k, g in enumerate(got))
        assert gpu.load().gf_release_device_cache(-1) == 0
