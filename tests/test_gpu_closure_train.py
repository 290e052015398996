"""Training of the p = 2, 256-unit closure at batch sizes around its tiles
(32 samples a workgroup, operands padded to 128 samples).

The reference is the layer-by-layer gradient (ldg_closure_gradient, itself
checked against numpy) and Adam in float64 numpy.  Every step starts from the
parameters the library holds, so differences do not accumulate: what is left
is the order of FP32 sums over the batch and the rounding of the FP32 moments.
Tolerances are those of the full-batch Adam test; the losses are sums of the
same FP32 squares, one rounding (6e-8) each: 1e-6.
"""
import numpy as np
import pytest

from ldg_amd import closure as C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 31, 33, 128, 129, 300])
def test_steps_match_gradient_and_adam(batch):
    steps, lr, b1, b2, eps = 3, 1e-3, 0.9, 0.999, 1e-8
    rng = np.random.default_rng(batch)
    c = C.Closure(2, 256, batch, seed=5)
    c.add_samples(rng.standard_normal((batch, c.nin)).astype(np.float32),
                  rng.standard_normal((batch, c.nout)).astype(np.float32))
    X, T = c.get_samples()
    probe = C.Closure(2, 256, 0, seed=0)
    m = np.zeros(c.get()[0].size)
    v = np.zeros_like(m)
    for t in range(1, steps + 1):
        before = c.get()[0]
        probe.set(before)
        g, loss = probe.gradient(X, T)
        g = g.astype(np.float64)
        m = b1 * m + (1 - b1) * g
        v = b2 * v + (1 - b2) * g * g
        ref = -lr * (m / (1 - b1 ** t)) / (np.sqrt(v / (1 - b2 ** t)) + eps)
        losses = c.train(1, batch=batch, lr=lr, val_fraction=0.0, seed=t)
        step = c.get()[0].astype(np.float64) - before
        err = np.abs(step - ref)
        print(f"batch {batch} step {t}: max |step| {np.abs(ref).max():.3e}, median error {np.median(err):.3e}",
              flush=True)
        assert abs(losses[0, 0] - loss) <= 1e-6 * loss
        assert losses[0, 1] == 0.0
        assert np.median(err) <= 1e-3 * lr
        assert np.quantile(err, 0.999) <= 5e-2 * np.abs(ref).max()
    probe.close()
    c.close()


def test_every_sample_enters_the_losses_once():
    """A learning rate that moves no parameter: training and hold-out losses
    together are the loss of all samples, whatever the permutation.  315
    training samples in 7 batches of 45, 185 held out in 4 batches and 5."""
    n, batch = 500, 45
    rng = np.random.default_rng(8)
    c = C.Closure(2, 256, n, seed=6)
    c.add_samples(rng.standard_normal((n, c.nin)).astype(np.float32),
                  (1.0 + rng.standard_normal((n, c.nout)) * rng.uniform(0.1, 3.0, (n, 1))).astype(np.float32))
    X, T = c.get_samples()
    _, loss = c.gradient(X, T)
    for tl, vl in c.train(2, batch=batch, lr=1e-30, val_fraction=0.37, seed=4):
        assert vl > 0.0
        assert abs((315 * tl + 185 * vl) / n - loss) <= 1e-6 * loss
    c.close()
