"""A frequency that is not a number adds nothing to the joint spectrum, in
either population, with either sign and whatever the sample sizes: the
spectrum is that of the other mutations, which the CPU oracle gives."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,nb", [(1, 1), (40, 40), (63, 63), (64, 40)])
def test_nan_frequencies_add_nothing(gpu, oracle, na, nb):
    rng = np.random.default_rng(na)
    M = 200
    fa, fb = rng.uniform(0, 1, (2, M)).astype(np.float32)
    nan = np.array([0x7fc00000, 0xffc00000, 0x7f800001, 0xff800001], np.uint32).view(np.float32)
    gone = np.zeros(M, bool)
    for k in range(4):
        fa[7 + k], fb[90 + k], fa[150 + k], fb[150 + k] = nan[k], nan[k], nan[k], nan[3 - k]
        gone[[7 + k, 90 + k, 150 + k]] = True
    fa[12:18] = [0.0, -0.0, 1.0, 1.5, -np.inf, np.inf]        # still lost, fixed
    fb[18:24] = fa[12:18]
    g = gpu.joint_site_frequency_spectrum(fa, fb, na, nb, 1e6)
    o = oracle.joint_site_frequency_spectrum(fa[~gone], fb[~gone], na, nb, 1e6 - gone.sum())
    assert np.array_equal(g.view(np.uint32), o.view(np.uint32))
