"""Whole training runs of the con2prim guess against a NumPy Adam loop."""
import numpy as np
import pytest

import mlp_ref
from helpers import progress

pytestmark = pytest.mark.gpu
G = 4.0 / 3.0
M64 = (1 << 64) - 1


def _splitmix(x):
    x = (x + 0x9E3779B97F4A7C15) & M64
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & M64
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & M64
    return x ^ (x >> 31)


def _adam(X, T, params, kw, dtype, fault=None):
    """(parameters, loss curve).  Sample s of step k is the valid pair
    splitmix64(seed ^ (k 0x100000001B3 + s)) mod n; the rate falls by a cosine
    from lr to lr_min; curve[k] is the loss before step k's update.  fault: a
    planted mistake."""
    w = params.astype(dtype)
    m, v = np.zeros_like(w), np.zeros_like(w)
    curve = []
    steps, b1, b2 = kw["steps"], kw["beta1"], kw["beta2"]
    for k in range(steps):
        at = [_splitmix(kw["seed"] ^ ((k * 0x100000001B3 + s) & M64)) % len(X) for s in range(kw["batch"])]
        loss, g = mlp_ref.loss_grad(w, X[at], T[at], w1=kw["w_out1"], qat=False, q_ref=kw["q_ref"], dtype=dtype)
        curve.append(loss)
        if fault == "last update dropped" and k == steps - 1:
            break
        m = b1 * m + (1 - b1) * g
        v = b2 * v + (1 - b2) * g * g
        j = k + 1 if fault == "rate of the next step" else k
        t = k + 2 if fault == "bias correction of the next step" else k + 1
        lr = kw["lr_min"] + 0.5 * (kw["lr"] - kw["lr_min"]) * (1 + np.cos(np.pi * j / steps))
        before = w
        w = w - lr * (m / (1 - b1 ** t)) / (np.sqrt(v / (1 - b2 ** t)) + kw["eps"])
    if fault == "buffer of the step before":
        w = before
    if fault == "loss curve shifted":
        curve = curve[1:] + curve[:1]
    return w.astype(np.float64), np.array(curve, np.float64)


@pytest.mark.parametrize("batch", [1, 40, 200, 8192])
@pytest.mark.parametrize("steps", [1, 2, 3, 4])
def test_training_is_adam(steps, batch):
    """Parameters and every entry of the loss curve after 1 to 4 steps, for
    batches of fewer samples than slices, of unequal slices and of many
    samples a slice.  Tolerance: 20 times what FP32 arithmetic changes in the
    NumPy loop itself, and at least 32 roundings of an FP32 parameter or loss of
    that size; a mistake in the steps' order, rates, corrections or buffers is
    ten times that or more (each is planted in the loop)."""
    from verona_amd.c2p import Con2PrimBatch, c4_states
    progress(f"adam steps={steps} batch={batch}")
    kw = dict(steps=steps, batch=batch, lr=3e-2, lr_min=1e-3, beta1=0.9, beta2=0.99, eps=1e-3, w_out1=0.7, q_ref=0.5,
              seed=11)
    U, P = c4_states(5000, seed=9, gamma=G)
    params = mlp_ref.he_init(13)
    with Con2PrimBatch(5000, G) as cp:
        X, T, ok = cp.features(U, P)
        curve, _ = cp.train(U, P, init=params, qat=False, **kw)
        got = cp.get_params().astype(np.float64)
    X, T = X[ok], T[ok]
    want, loss = _adam(X, T, params, kw, np.float64)
    want32, loss32 = _adam(X, T, params, kw, np.float32)
    tol = max(20 * np.abs(want32 - want).max(), 32 * 2.0**-24 * np.abs(want).max())
    ltol = np.maximum(20 * np.abs(loss32 - loss), 32 * 2.0**-24 * loss)
    progress(f"  params off by {np.abs(got - want).max():.1e} of {tol:.1e}, loss {np.abs(curve - loss).max():.1e} of {ltol.max():.1e}")
    assert np.abs(got - want).max() <= tol
    assert (np.abs(curve - loss) <= ltol).all()
    for fault in ("last update dropped", "buffer of the step before", "rate of the next step",
                  "bias correction of the next step"):
        assert np.abs(_adam(X, T, params, kw, np.float64, fault)[0] - want).max() > 10 * tol, fault
    if steps > 1:
        assert (np.abs(_adam(X, T, params, kw, np.float64, "loss curve shifted")[1] - loss) > 10 * ltol).any()
