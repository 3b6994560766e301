"""The order in which an epoch visits the training points: the device finds each
entry of the seeded shuffle on its own; here it is the loop it stands for
(splitmix64 draws, Fisher-Yates from the last entry down).

The order shows in the trained network alone.  Two seeds give two orders; the
points are laid out for each so that training meets the same sequence, and the
same sums make the same network bit for bit.  Two epochs are one epoch, then one
from the state that the first leaves.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from goma_amd import capi  # noqa: E402

STEP, MASK = 0x9E3779B97F4A7C15, (1 << 64) - 1


def _order(n, seed):
    p, s = list(range(n)), seed
    for i in range(n - 1, 0, -1):
        s = (s + STEP) & MASK
        z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & MASK
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & MASK
        j = (z ^ (z >> 31)) % (i + 1)
        p[i], p[j] = p[j], p[i]
    return np.array(p)


# one point, two, a batch and its neighbours, several workgroups, many batches
@pytest.mark.parametrize("n,batch", [(1, 128), (2, 128), (128, 128), (129, 128), (257, 128),
                                     (1000, 128), (40001, 8192)])
def test_training_order(n, batch):
    print(f"[case] training order n {n} batch {batch}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    t = rng.standard_normal((n, 2)).astype(np.float32)
    m = (rng.uniform(size=(n, 2)) > 0.2).astype(np.float32)
    out = []
    for seed in (9, MASK - 5):
        net = capi.Mlp(3, 2, hidden=1, width=64, seed=5)
        at = np.empty(n, np.int64)
        at[_order(n, seed)] = np.arange(n)  # the point met k-th is row k of x
        net.set_data(x[at], t[at], m[at])
        net.train(epochs=1, batch=batch, lr=1e-2, lr_final=1e-2, seed=seed)
        out.append(net.get_params())
        net.close()
    assert np.isfinite(out[0]).all() and np.array_equal(out[0], out[1])


def test_epochs_go_on_from_the_last_draw():
    print("[case] training order over epochs", flush=True)
    n, out = 700, []
    rng = np.random.default_rng(3)
    data = (rng.uniform(0, 1, (n, 3)).astype(np.float32),
            rng.standard_normal((n, 2)).astype(np.float32), np.ones((n, 2), np.float32))
    for runs in ([(2, 9)], [(1, 9), (1, (9 + (n - 1) * STEP) & MASK)]):
        net = capi.Mlp(3, 2, hidden=1, width=64, seed=5)
        net.set_data(*data)
        for epochs, seed in runs:
            net.train(epochs=epochs, batch=128, lr=1e-2, lr_final=1e-2, seed=seed)
        out.append(net.get_params())
        net.close()
    assert np.array_equal(out[0], out[1])
