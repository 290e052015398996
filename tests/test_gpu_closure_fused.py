"""The fused closure inference forms the nodal gradient itself: its correction
on ragged meshes (element counts around and between multiples of the 32 of a
workgroup, unequal axes) against the network evaluated layer by layer on the
features of the state and of ldg_rhs's gradient output.

Tolerance 1e-4 of the largest correction, as for the same comparison in
test_gpu_closure.py: features equal to FP64 (FP32) rounding may round to
neighbouring BF16 values on the host and on the device in a few places.
"""
import numpy as np
import pytest

import ldg_amd
from ldg_amd import closure as C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [ldg_amd.LDG_FP64, ldg_amd.LDG_MIXED])
@pytest.mark.parametrize("mesh", [(3, 3, 3), (4, 4, 4), (3, 11, 5), (13, 5, 3)])
def test_fused_inference_matches_layers_on_ragged_meshes(mesh, precision):
    plain = ldg_amd.LDG(2, *mesh, precision=precision)
    corr = ldg_amd.LDG(2, *mesh, precision=precision)
    c = C.Closure(2, 256, 0, seed=8)
    rng = np.random.default_rng(5)
    nin, nout = c.nin, c.nout
    plain.initial_condition()
    u = plain.get_state()
    u[:, 1:4] += 0.05 * rng.standard_normal(u[:, 1:4].shape)       # every gradient component differs
    k0, du = plain.rhs(u, want_du=True)
    K = u.shape[0]
    w = u.copy()
    w[:, 0] -= 1.0
    w[:, 4] -= (1.0 / 0.1) ** 2 / 1.4 / (1.4 - 1.0)
    x = np.concatenate([w.reshape(K, -1), np.transpose(du, (1, 0, 2, 3)).reshape(K, -1)], axis=1)
    norm = np.concatenate([x.mean(0), 1 / (x.std(0) + 1e-3), rng.standard_normal(nout), rng.uniform(0.5, 2.0, nout)])
    norm = norm.astype(np.float32)
    c.set(norm=norm)
    C.attach(corr, c, 1e30)
    k1 = corr.rhs(u)
    assert C.gated(corr) == (0, K)
    X = ((x - norm[:nin]) * norm[nin:2 * nin]).astype(np.float32)
    expect = (c.forward(X).astype(np.float64) * norm[2 * nin + nout:] + norm[2 * nin:2 * nin + nout]).reshape(k0.shape)
    e = float(np.max(np.abs(k1 - k0 - expect)) / np.max(np.abs(expect)))
    print("mesh", mesh, "relative error", e, flush=True)
    assert e <= 1e-4
