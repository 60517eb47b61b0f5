"""Fixed mutations that a model loses again: with s(1) <= -1 Eq. 13 is 0/0 at
a frequency of 1, whose draw is 0 in the oracle.  Runs that keep fixed
mutations (preserved, or never compacted), go to such a model at generation
101 and may or may not start a launch there, against the CPU oracle bit for
bit."""
import numpy as np
import pytest

from parallelpopgen_amd import scenarios as S
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slope,intercept", [(0.0, -1.0), (0.0, -1.5), (-1.1, 0.05)])
@pytest.mark.parametrize("interval,preserve", [(0, 0), (35, 30)])
@pytest.mark.parametrize("sample,kpl", [(0, 0), (100, 0), (100, 7)])
def test_fixed_under_lethal_selection(gpu, oracle, slope, intercept, interval, preserve, sample, kpl):
    d = S.constant(N=200, L=2e7, G=200, compact_interval=interval, preserve_every=preserve, sample_every=sample)
    d.params["sel_intercept"][1:101] = 0.05
    d.params["sel_slope"][101:], d.params["sel_intercept"][101:] = slope, intercept
    gpu.set_generations_per_launch(kpl)
    try:
        a = gpu.run(d)
    finally:
        gpu.set_generations_per_launch(0)
    o = oracle.run(d)
    if sample:
        assert np.sum(o["samples"][1]["freq"] >= 1.0) > 0     # fixed at generation 100
    assert np.sum(o["samples"][-1]["freq"] >= 1.0) == 0
    assert_same(a, o, (slope, intercept, interval, sample, kpl))
