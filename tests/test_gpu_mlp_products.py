"""The warm-start network's products at the edges of their 16- and 32-wide tiles and
16-index stages, against the float64 oracle."""
import numpy as np
import pytest

import oracle.warmstart as W

pytestmark = pytest.mark.gpu
EPS = 2.0**-24


@pytest.mark.parametrize("batch,K,N", [(1, 1, 1), (3, 15, 17), (16, 16, 16), (17, 31, 33), (40, 129, 65),
                                       (256, 200, 256), (130, 257, 20), (1030, 40, 1025)])
def test_one_layer(itcpd, batch, K, N):
    """Y = X W + b within (K + 2) eps of the sums of magnitudes; dW = X^T dZ and db = 1^T dZ
    within (batch + 4) eps of theirs plus what Y's error carries through dZ."""
    rng = np.random.default_rng(1)
    X = rng.standard_normal((batch, K)).astype(np.float32)
    Yt = rng.standard_normal((batch, N)).astype(np.float32)
    par = rng.standard_normal(K * N + N).astype(np.float32)
    with itcpd.MLP([K, N], batch_cap=batch) as net:
        net.set_params(par)
        Y = net.forward(X)
        g, _ = net.gradients(X, Yt)
    Wm, b = par[:K * N].reshape(K, N).astype(np.float64), par[K * N:].astype(np.float64)
    Xd = X.astype(np.float64)
    ref = Xd @ Wm + b
    ebound = (K + 2) * EPS * (np.abs(Xd) @ np.abs(Wm) + np.abs(b))
    assert (np.abs(Y - ref) / ebound).max() <= 1.0
    dZ = (ref - Yt) / batch
    edz = (ebound + 3 * EPS * (np.abs(ref) + np.abs(Yt))) / batch
    for got, lhs in ((g[:K * N].reshape(K, N), Xd), (g[K * N:], np.ones(batch))):
        bound = (batch + 4) * EPS * (np.abs(lhs).T @ np.abs(dZ)) + 1.1 * (np.abs(lhs).T @ edz)
        assert (np.abs(got - lhs.T @ dZ) / bound).max() <= 1.0


@pytest.mark.parametrize("widths,batch", [([5, 17, 3], 9), ([33, 64, 31, 16], 47), ([64, 1030, 1030, 8], 1030)])
def test_hidden_layers(itcpd, widths, batch):
    """The gated backward product, with both tile sizes: relative errors of a few hundred
    float32 roundings (1e-5), as the network's other tests.  A gate is a step function of a
    rounded sum, so the oracle takes the gates that the same products give layer by layer;
    they may differ from float64's only where the sum is zero to its own rounding."""
    rng = np.random.default_rng(2)
    X = rng.standard_normal((batch, widths[0])).astype(np.float32)
    Yt = rng.standard_normal((batch, widths[-1])).astype(np.float32)
    mask = (rng.random((batch, widths[-1])) < 0.8).astype(np.float32)
    with itcpd.MLP(widths, batch_cap=batch, seed=3) as net:
        par = net.params()
        g, loss = net.gradients(X, Yt, mask)
    Ws, bs = W.unpack(par, widths)
    gates, H32, H = [], X, [X.astype(np.float64)]
    for Wl, b in zip(Ws[:-1], bs[:-1]):
        with itcpd.MLP(list(Wl.shape), batch_cap=batch) as one:
            one.set_params(np.concatenate([Wl.ravel(), b]).astype(np.float32))
            H32 = np.maximum(one.forward(H32), 0)
        Z = H[-1] @ Wl + b
        gate = H32 > 0
        bound = 8 * (Wl.shape[0] + 2) * EPS * (np.abs(H[-1]) @ np.abs(Wl) + np.abs(b))
        assert np.all((np.abs(Z) <= bound)[gate != (Z > 0)])
        gates.append(gate)
        H.append(Z * gate)
    Y = H[-1] @ Ws[-1] + bs[-1]
    D = mask * (Y - Yt)
    dZ, parts = D / batch, []
    for l in range(len(Ws) - 1, -1, -1):
        parts = [(H[l].T @ dZ).ravel(), dZ.sum(axis=0)] + parts
        if l:
            dZ = (dZ @ Ws[l].T) * gates[l - 1]
    ref = np.concatenate(parts)
    ref_loss = 0.5 * float(np.sum(D * D)) / batch
    assert abs(loss - ref_loss) <= 1e-5 * ref_loss
    assert np.linalg.norm(g - ref) <= 1e-5 * np.linalg.norm(ref)
