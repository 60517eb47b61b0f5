"""The one-kernel network of prediction (k_mlp) at the edges of its tiles and
of the rule that picks them: 32-row tiles while every member's tiles fit one
a CU, 64-row tiles beyond, ragged counts, ensembles whose tiles do not divide
over the 8 XCDs, and weights replaced between calls.  Rows do not depend on
the rows beside them: each prediction of a batch equals, bit for bit, that
input's in another batch; the logits are checked against the float64 oracle
with the same bfloat16 rounding points (tolerance as for the training
products: one bfloat16 rounding on the other side of a tie moves a logit by
less than 1e-2 of their RMS)."""
import numpy as np
import pytest

from oracle import surrogate_oracle as SO
from parallelpopgen_amd import surrogate as SG

pytestmark = pytest.mark.gpu


def inputs(n, seed):
    return np.random.default_rng(seed).uniform(-1, 1, (n, 6)).astype(np.float32)


@pytest.mark.parametrize("E", [1, 3, 5])
@pytest.mark.parametrize("n", [1, 31, 33, 64, 65, 2049, 8257])
def test_rows_are_independent(E, n):
    net = SG.Network(ensemble=E, seed=30 + E)
    x = inputs(n, n)
    sfs, tot, dis = net.predict(x)
    big = np.concatenate([x[::-1], inputs(20000, 1)])      # other tiles, other neighbours
    s2, t2, d2 = net.predict(big)
    assert np.array_equal(sfs, s2[:n][::-1]) and np.array_equal(tot, t2[:n][::-1]) and np.array_equal(dis, d2[:n][::-1])
    net.close()


@pytest.mark.parametrize("n", [64, 4096, 8192])
def test_logits_match_oracle_after_new_weights(n):
    net = SG.Network(ensemble=2, seed=40)
    x = inputs(n, 2)
    net.forward(x[:64])
    p = SG.Network(ensemble=2, seed=41).get_params()
    net.set_params(p)                                       # the packed copy has to follow
    L = net.forward(x)
    rows = np.r_[0:64, n - 64:n]
    for e in range(2):
        _, _, ref = SO.forward(p[e].astype(np.float64), x[rows].astype(np.float64))
        err = np.abs(L[e][rows, :SO.OUT] - ref[:, :SO.OUT]).max()
        assert err <= 1e-2 * np.sqrt(np.mean(ref[:, :SO.OUT] ** 2)), (e, err)
        assert np.all(L[e][:, SO.OUT:] == 0.0)
    y = np.full((64, SG.NBINS), 1.0 / SG.NBINS, np.float32)
    net.train(x[:64], y, np.zeros(64, np.float32), epochs=1, batch=64, lr=0.05, shuffle=False)
    q = net.get_params()
    _, _, ref = SO.forward(q[0].astype(np.float64), x[:64].astype(np.float64))
    assert np.abs(net.forward(x[:64])[0][:, :SO.OUT] - ref[:, :SO.OUT]).max() <= 1e-2 * np.sqrt(np.mean(ref[:, :SO.OUT] ** 2))
    net.close()
