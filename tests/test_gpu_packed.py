"""Slots that hold something gathered from several tiles (gf_packed_drift.hpp)
against the CPU oracle, bit for bit: launches of more than 16,384 tiles (4.2e6
slots, most of them new), with preserved mutations, samples, launches that do
not compact, selection without and with a slope, and migration."""
import numpy as np
import pytest

from parallelpopgen_amd import scenarios as S
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,L,s,slope,interval,preserve,kpl", [
    (2, 1.5e11, 0.0, 0.0, 9, 6, 0),
    (2, 1.5e11, -0.01, 0.0, 12, 0, 7),     # every other launch does not compact
    (3, 1.0e11, 0.002, 0.0, 7, 10, 0),
    (4, 0.8e11, -0.01, 0.02, 0, 5, 0),     # never compacts
    (4, 0.8e11, -0.01, 0.0, 11, 11, 0),
])
def test_packed_against_oracle(gpu, oracle, P, L, s, slope, interval, preserve, kpl):
    d = S.constant(N=400, L=L, G=14, s=s, h=0.3, F=0.1, P=P, m=0.01, compact_interval=interval, preserve_every=preserve,
                   sample_every=13)
    d.params["sel_slope"] = slope
    d.params["N"][8:, P - 1] = 0     # the last population ends
    d.migration[8:] = 0
    for t in range(8, 15):
        d.migration[t, :P - 1, :P - 1] = S.migration_constant_equal(0.01, P - 1)
    gpu.set_generations_per_launch(kpl)
    try:
        a = gpu.run(d)
    finally:
        gpu.set_generations_per_launch(0)
    assert_same(a, oracle.run(d), (P, interval))
