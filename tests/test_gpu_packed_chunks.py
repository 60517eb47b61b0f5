"""The packed drift of several populations with its largest chunks, eight
tiles, which it takes from 65,536 tiles (1.7e7 slots) on: against the CPU
oracle bit for bit, with preserved mutations, and with selection that has a
slope and launches that do not compact."""
import pytest

from parallelpopgen_amd import scenarios as S
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,L,slope,interval,preserve,kpl", [
    (2, 6.5e11, 0.0, 6, 5, 0),
    (3, 4.4e11, 0.02, 8, 0, 5),
])
def test_eight_tiles_a_chunk(gpu, oracle, P, L, slope, interval, preserve, kpl):
    d = S.constant(N=400, L=L, G=9, s=-0.01, h=0.3, F=0.1, P=P, m=0.01, compact_interval=interval, preserve_every=preserve)
    d.params["sel_slope"][1:] = slope
    d.params["sel_intercept"][0] = 0.0
    gpu.set_generations_per_launch(kpl)
    oracle.set_threads(16)
    try:
        a, o = gpu.run(d), oracle.run(d)
    finally:
        gpu.set_generations_per_launch(0)
        oracle.set_threads(1)
    assert o["live"][0] > 65536 * 200
    assert_same(a, o, (P, interval))
