"""The two training kernels (k_train_rows, k_train_weights) where their tiles
and orders can go wrong: the smallest batch (one round of the contraction's
prefetch), batches past one round with an odd number of 64-row pieces, member
counts that do not divide over the 8 XCDs, rows gathered through an order, and
the padding of the network (inputs 6..63, outputs 100..127).  Gradients
against the float64 oracle with the same bfloat16 rounding points (3e-2 in
relative L2 norm: a bfloat16 rounding on the other side of a tie)."""
import numpy as np
import pytest

from oracle import surrogate_oracle as SO
from parallelpopgen_amd import surrogate as SG

pytestmark = pytest.mark.gpu


def data(n, seed):
    rng = np.random.default_rng(seed)
    return (rng.uniform(-1, 1, (n, 6)).astype(np.float32), rng.dirichlet(np.ones(SO.NBINS) * 0.5, n).astype(np.float32),
            rng.normal(0, 1, n).astype(np.float32))


@pytest.mark.parametrize("E,B", [(1, 64), (5, 320), (3, 1088)])
def test_gradients(E, B):
    net = SG.Network(ensemble=E, seed=50)
    x, y, t = data(B, B)
    loss, g = net.gradients(x, y, t, w_tot=0.7)
    p = net.get_params()
    offs, total = SO.layout()
    for e in (0, E - 1):
        lo, go = SO.loss_and_grads(p[e].astype(np.float64), x.astype(np.float64), y.astype(np.float64),
                                   t.astype(np.float64), 0.7)
        assert abs(loss[e] - lo) <= 1e-3 * abs(lo)
        for l, (w, b) in enumerate(offs):
            for a, n in ((w, SO.INS[l] * SO.OUTS[l]), (b, SO.OUTS[l])):
                d = np.linalg.norm(g[e, a:a + n] - go[a:a + n]) / np.linalg.norm(go[a:a + n])
                assert d < 3e-2, (e, l, d)
        w0 = g[e, offs[0][0]:offs[0][0] + 512 * 64].reshape(512, 64)
        w4 = g[e, offs[4][0]:offs[4][0] + 128 * 512].reshape(128, 512)
        assert np.all(w0[:, 6:] == 0) and np.all(w4[100:] == 0)
    net.close()


def test_order_is_a_gather():
    """visiting rows through an order equals, bit for bit, storing them in that order"""
    x, y, t = data(640, 3)
    o = np.random.default_rng(4).permutation(640)
    a, b = SG.Network(ensemble=3, seed=51), SG.Network(ensemble=3, seed=51)
    order = np.ascontiguousarray(o[None, :], np.int32)
    loss = np.empty(1, np.float32)
    from parallelpopgen_amd import capi
    capi.check(a.lib.gf_sg_train(a.h, SG._p(x), SG._p(y), SG._p(t), 640, 1, 128, 1e-3, 0.5, SG._p(order), SG._p(loss)))
    b.train(x[o], y[o], t[o], epochs=1, batch=128, lr=1e-3, w_tot=0.5, shuffle=False)
    assert np.array_equal(a.get_params().view(np.uint32), b.get_params().view(np.uint32))
    a.close()
    b.close()
