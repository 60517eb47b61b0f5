"""The wave form of the joint spectrum (samples of up to 63 chromosomes) at
its edges, against the CPU oracle bit for bit: sample sizes at and past the
limit of either population, counts around its batches of 32 mutations, and
frequencies whose products reach 1 (0, 1, and tiny ones, whose probability of
no copy rounds to 1)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,nb", [(1, 1), (63, 63), (63, 2), (64, 63), (63, 64), (31, 40)])
@pytest.mark.parametrize("M", [1, 31, 32, 33, 5001])
def test_joint_edges(gpu, oracle, na, nb, M):
    rng = np.random.default_rng(M + na)
    fa = np.exp(rng.uniform(-12, 0, M)).astype(np.float32)
    fb = np.clip(fa * np.exp(rng.normal(0, 1, M)), 0, 1).astype(np.float32)
    special = np.array([0.0, 1.0, 1e-9, 1e-30, 0.99999994, 0.5], np.float32)
    for k in range(min(M, 36)):
        fa[M - 1 - k], fb[M - 1 - k] = special[k % 6], special[k // 6]
    g = gpu.joint_site_frequency_spectrum(fa, fb, na, nb, 1e6)
    o = oracle.joint_site_frequency_spectrum(fa, fb, na, nb, 1e6)
    assert np.array_equal(g.view(np.uint32), o.view(np.uint32))
