"""Sample spectra of more than a million chromosomes, whose float
log-binomial table is off by more than 88: the levels whose exponential
overflows hold the largest sum, 2^64 units of 2^-32, and the others their own
term.  One mutation, so a level is one term; the terms from the oracle's log
and exp."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,p", [(1_500_000, 0.25), (1_500_000, 0.3), (2_000_001, 0.4), (2_000_001, 0.45)])
def test_overflowing_levels(gpu, oracle, n, p):
    f = np.float32(p)
    half = n // 2 + 1 if n % 2 == 0 else (n + 1) // 2
    k = np.arange(1, half, dtype=np.float32)
    lc = np.zeros(half, np.float32)
    lc[1:] = np.cumsum(oracle.log_f(((np.float32(n) + np.float32(1)) - k) / k), dtype=np.float32)
    lp, lq = oracle.log_f(np.array([f, np.float32(1) - f], np.float32))
    k = np.arange(n + 1)
    t = (np.where(k < half, lc[np.minimum(k, half - 1)], lc[np.minimum(n - k, half - 1)]) +
         k.astype(np.float32) * lp) + (n - k).astype(np.float32) * lq
    km = int(np.float32(n + 1) * f)
    below = t < -24.0                           # the levels from the mode out to the first such one
    lo = np.nonzero(below[:km])[0]
    hi = np.nonzero(below[km:])[0]
    lo = lo[-1] + 1 if len(lo) else 0
    hi = km + hi[0] if len(hi) else n + 1
    seen = (k >= lo) & (k < hi) & (t >= -23.0)
    assert t[seen].max() > 90.0                 # exp overflows
    term = np.where(seen, oracle.exp_f(t), np.float32(0)).astype(np.float32)
    units = np.minimum(term.astype(np.float64) * 2.0 ** 32, 2.0 ** 64)
    want = (np.floor(units) / 2.0 ** 32).astype(np.float32)
    got = gpu.site_frequency_spectrum(np.array([f]), n, 1e6)
    bad = np.nonzero(got[1:] != want[1:n])[0]
    assert bad.size == 0, (bad.size, bad[:3] + 1, got[1:][bad[:3]], want[1:n][bad[:3]], t[1:n][bad[:3]])
