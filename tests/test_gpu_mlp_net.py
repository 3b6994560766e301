"""The whole-network kernels (one tile of points through every layer) at the
edges of their tiles and of the networks they take, against the CPU oracle.

Bars as for the layer-by-layer kernels: the GPU and the oracle round at the
same points, so the loss agrees to 1e-4 and each layer's gradient to 5e-3 (rare
BF16 rounding flips).  Prediction takes the forward sums of training: its loss
agrees to the FP32 rounding of the errors, under 1e-6.  Large and small batches
go through different tiles of the same sums: equal bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from goma_amd import capi  # noqa: E402
from oracle import MlpOracle  # noqa: E402


def _pair(n_in, n_out, hidden, width):
    sh, sc = [0.5] * n_in, [2.0] * n_in
    net = capi.Mlp(n_in, n_out, hidden=hidden, width=width, seed=5, in_shift=sh, in_scale=sc)
    rng = np.random.default_rng(width + hidden)
    p = net.get_params() + 0.02 * rng.standard_normal(net.num_params).astype(np.float32)
    net.set_params(p)
    return net, MlpOracle(n_in, n_out, hidden, width, in_shift=sh, in_scale=sc), p, rng


# widths of each wave split; one hidden layer; the deepest network whose
# activations fit in LDS at width 256 and the first that does not; a width
# beyond the whole-network kernels
@pytest.mark.parametrize("n_in,n_out,hidden,width,npts", [
    (1, 1, 1, 64, 1), (3, 4, 2, 64, 33), (8, 8, 1, 128, 127), (4, 5, 3, 192, 129), (4, 5, 4, 256, 31),
    (3, 4, 4, 128, 513), (2, 3, 9, 256, 40), (2, 3, 10, 256, 40), (3, 4, 2, 320, 65)])
def test_gradient_and_prediction(n_in, n_out, hidden, width, npts):
    print(f"[case] net {n_in}-{width}x{hidden}-{n_out} npts {npts}", flush=True)
    net, o, p, rng = _pair(n_in, n_out, hidden, width)
    x = rng.uniform(0, 1, (npts, n_in)).astype(np.float32)
    t = rng.standard_normal((npts, n_out)).astype(np.float32)
    m = (rng.uniform(size=(npts, n_out)) > 0.2).astype(np.float32)
    m[0, 0] = 1.0
    lg, gg = net.loss_grad(x, t, m)
    lo, go = o.loss_grad(p, x, t, m, quant=True)
    assert abs(lg - lo) <= 1e-4 * lo
    at, k = 0, n_in
    for n in [width] * hidden + [n_out]:
        a, at, k = at, at + n * k + n, n
        assert np.linalg.norm(gg[a:at] - go[a:at]) < 5e-3 * np.linalg.norm(go[a:at]), a
    # prediction and training run the same sums: the loss follows from the prediction
    y = net.predict(x).astype(np.float64)
    assert abs((m * (y - t) ** 2).sum() / (npts * n_out) - lg) <= 1e-6 * lg
    net.close()


@pytest.mark.parametrize("width", [64, 128, 192, 256])
def test_large_and_small_tiles_agree(width):
    print(f"[case] net tiles width {width}", flush=True)
    net, _, _, rng = _pair(4, 5, 2, width)
    n = 128 * 512 + 77  # the large tile's range, its last tile ragged
    x = rng.uniform(0, 1, (n, 4)).astype(np.float32)
    y = net.predict(x)
    parts = np.concatenate([net.predict(c) for c in np.split(x, [1, 32, 5000, 65000])])
    assert np.isfinite(y).all() and np.array_equal(y, parts)
    net.close()
