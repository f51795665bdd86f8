"""The network's two ways through the device have the same bits: a network that trains in three launches
and predicts in one (up to 256 features a layer), and the same network among 288 features a layer, the
further ones' weights and biases zero, which goes layer by layer. The zeros add nothing to any sum and
stay zero (their gradients are), so that gradients, loss, trained weights and predictions have to be
equal: over widths and depths, both splits of the weight gradients over the rows, and rows below and above
the 8192 that a bias sum takes in one round."""
import numpy as np
import pytest

from cfd_solver_withcuda_amd.surrogate import MLP

pytestmark = pytest.mark.gpu
WIDE = 288


def layers(n_in, width, depth, n_out):
    return [(width if k < depth else n_out, width if k else n_in) for k in range(depth + 1)]


def widened(W, b, small, wide):
    """The parameters among the wide network's zeros."""
    Ws, bs, ow, ob = [], [], 0, 0
    for (m, k), (M, K) in zip(small, wide):
        w = np.zeros((M, K), np.float32)
        w[:m, :k] = W[ow:ow + m * k].reshape(m, k)
        v = np.zeros(M, np.float32)
        v[:m] = b[ob:ob + m]
        Ws.append(w.ravel())
        bs.append(v)
        ow, ob = ow + m * k, ob + m
    return np.concatenate(Ws), np.concatenate(bs)


@pytest.mark.parametrize("n_in,width,depth,n_out,rows", [
    (4, 256, 6, 4, 1024), (4, 256, 6, 4, 8704), (4, 32, 2, 4, 512), (3, 64, 1, 1, 1536), (7, 160, 2, 5, 16384),
    (31, 100, 3, 32, 9216), (4, 192, 15, 4, 512)])
def test_three_launches_and_layer_by_layer(n_in, width, depth, n_out, rows):
    print(f"case {n_in} -> {depth} x {width} -> {n_out}, {rows} rows", flush=True)
    r = np.random.default_rng(width + depth)
    feat = r.uniform(-1, 1, (rows, n_in)).astype(np.float32)
    targ = (1.5 + np.sin(feat @ r.uniform(-2, 2, (n_in, n_out)))).astype(np.float32)
    small, wide = layers(n_in, width, depth, n_out), layers(n_in, WIDE, depth, n_out)
    a, b = MLP(n_in, width, depth, n_out, max_rows=rows, seed=3), MLP(n_in, WIDE, depth, n_out, max_rows=rows, seed=4)
    for m in (a, b):
        m.fit_normalization(feat, targ)
    W = a.get_params()[0]
    bias = r.uniform(-0.1, 0.1, sum(m for m, _ in small)).astype(np.float32)
    a.set_params(W, bias)
    b.set_params(*widened(W, bias, small, wide))
    la, gW, gb = a.gradients(feat, targ)
    lb, hW, hb = b.gradients(feat, targ)
    eW, eb = widened(gW, gb, small, wide)
    assert np.array_equal(eW, hW) and np.array_equal(eb, hb) and la == lb
    assert np.count_nonzero(gW) > len(gW) // 2
    for n in (1, 63, rows, rows + 65):
        f = r.uniform(-1, 1, (n, n_in)).astype(np.float32)
        assert np.array_equal(a.predict(f), b.predict(f)), n
    for launch in ("kernels", "graph"):
        hist = []
        for m in (a, b):
            m.set_launch(launch)
            hist.append(m.train(feat, targ, steps=5, batch=rows, lr=2e-3, lr_final=1e-3, seed=2, log_every=1))
        assert np.array_equal(*hist), launch
        W, bias = a.get_params()
        eW, eb = widened(W, bias, small, wide)
        hW, hb = b.get_params()
        assert np.array_equal(eW, hW) and np.array_equal(eb, hb), launch
