"""Networks of one width and different depths, trained from two threads.

Both go through the same training kernel, with different amounts of LDS (five
and nine layers of 256 in a tile): each must end with the parameters that it
reaches alone, bit for bit.
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from goma_amd import capi  # noqa: E402

DEPTHS = (4, 9)


def _train(hidden, out):
    net = capi.Mlp(4, 5, hidden=hidden, width=256, seed=hidden, in_shift=[0.5] * 4, in_scale=[2.0] * 4)
    rng = np.random.default_rng(hidden)
    x = rng.uniform(0, 1, (4096, 4)).astype(np.float32)
    t = rng.standard_normal((4096, 5)).astype(np.float32)
    net.set_data(x, t, np.ones_like(t))
    net.train(epochs=20, batch=1024, lr=1e-3, lr_final=1e-4, seed=3)
    out[hidden] = net.get_params()
    net.close()


def test_two_depths_side_by_side():
    alone, beside = {}, {}
    for h in DEPTHS:
        print(f"[case] net 4-256x{h}-5 alone", flush=True)
        _train(h, alone)
    print("[case] both nets, two threads", flush=True)
    threads = [threading.Thread(target=_train, args=(h, beside)) for h in DEPTHS]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for h in DEPTHS:
        assert np.isfinite(alone[h]).all() and np.array_equal(alone[h], beside[h]), h
