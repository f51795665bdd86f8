"""The MLP's three-launch training step and its prediction over the shapes at which waves, tiles and
paddings change (outputs of one to eight blocks of 32, widths that are no multiple of 32, the
narrowest and the widest network that fits, one beyond it, one hidden layer), against the FP64
oracle with the device's BF16 rounding points."""
import numpy as np
import pytest

from cfd_solver_withcuda_amd.surrogate import MLP
from oracle.mlp_oracle import MLP as OMLP

pytestmark = pytest.mark.gpu


def data(n, n_in, n_out, seed):
    r = np.random.default_rng(seed)
    feat = r.uniform(-1, 1, (n, n_in)).astype(np.float32)
    w = r.uniform(-2, 2, (n_in, n_out))
    return feat, (1.5 + np.sin(feat @ w)).astype(np.float32)


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("n_in,width,depth,n_out,rows", [
    (4, 256, 6, 4, 1024), (4, 32, 2, 4, 512), (3, 64, 1, 1, 512), (4, 96, 3, 4, 1536), (4, 128, 4, 4, 512),
    (7, 160, 2, 5, 1024), (4, 192, 5, 4, 512), (4, 224, 2, 4, 512), (31, 100, 2, 32, 1024), (32, 250, 2, 3, 512),
    (4, 320, 2, 4, 512)])
def test_gradients_and_prediction_vs_oracle(n_in, width, depth, n_out, rows):
    print(f"case {n_in} -> {depth} x {width} -> {n_out}, {rows} rows", flush=True)
    feat, targ = data(rows, n_in, n_out, width)
    m = MLP(n_in, width, depth, n_out, max_rows=rows, seed=3)
    m.fit_normalization(feat, targ)
    W, b = m.get_params()
    b = np.random.default_rng(1).uniform(-0.1, 0.1, len(b)).astype(np.float32)
    m.set_params(W, b)
    o = OMLP(n_in, width, depth, n_out)
    norm = [a.astype(np.float64) for a in m.norm]
    args = (W.astype(np.float64), b.astype(np.float64))
    loss, gW, gb = m.gradients(feat, targ)
    oloss, ogW, ogb = o.loss_and_grads(*args, feat.astype(np.float64), targ.astype(np.float64), norm, bf16=True)
    # BF16 rounding flips where the FP32 sums and the oracle's FP64 sums round differently: the bounds
    # of the 6 x 256 network's test
    assert loss == pytest.approx(oloss, rel=2e-3)
    ow = ob = 0
    for k, n in o.dims:
        assert rel(gW[ow:ow + k * n], ogW[ow:ow + k * n]) < 3e-2 and rel(gb[ob:ob + n], ogb[ob:ob + n]) < 3e-2
        ow, ob = ow + k * n, ob + n
    for n in (1, 63, rows, rows + 65):  # beyond max_rows: more than one chunk
        f, _ = data(n, n_in, n_out, 5)
        want = o.predict(*args, f.astype(np.float64), norm, bf16=True)
        assert np.abs(m.predict(f) - want).max() <= 2e-2 * np.abs(want).max()
    # training moves the weights the way the gradients point, and lowers the loss
    hist = m.train(feat, targ, steps=60, batch=512, lr=2e-3, lr_final=1e-3, seed=2, log_every=59)
    assert np.all(np.isfinite(hist)) and hist[-1] < hist[0]
