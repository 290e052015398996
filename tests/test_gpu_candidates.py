"""Every kernel candidate (elements per workgroup, or a wave per variable)
gives the same right-hand side and state, bit by bit, whichever the
autotuner or the rule on element counts would take: set one by one through
libldg_test.so on meshes whose last workgroups are partial.  With the closure
attached the right-hand side kernel also adds the gated corrections.  The
energies sum per-workgroup partials, in another order: 1e-13."""
import ctypes
import os

import numpy as np
import pytest

import ldg_amd
from ldg_amd import closure as C
from test_zz_no_alloc import _hip, _noalloc_rhs

pytestmark = pytest.mark.gpu

PRECISIONS = [ldg_amd.LDG_FP64, ldg_amd.LDG_MIXED]


def _candidates():
    lib = ctypes.CDLL(os.path.join(os.path.dirname(ldg_amd.__file__), "libldg_test.so"))
    lib.ldg_test_set_candidates.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int]
    lib.ldg_test_set_candidates.restype = None
    return lib


def _noisy(g, seed):
    g.initial_condition()
    u = g.get_state()
    rng = np.random.default_rng(seed)
    for s, a in enumerate((1e-3, 2e-2, 2e-2, 2e-2, 1e-1)):
        u[:, s] += a * rng.standard_normal(u[:, s].shape)
    return u


def _answers(lib, g, u, grad, rhs):
    lib.ldg_test_set_candidates(g._h, grad, rhs)
    k = g.rhs(u)
    g.set_state(u)
    ke = g.step(1e-4, 3)
    return k, g.get_state(), ke


@pytest.mark.parametrize("precision", PRECISIONS)
@pytest.mark.parametrize("p", [1, 2, 3, 4, 5])
def test_candidates_agree_bitwise(p, precision):
    lib = _candidates()
    g = ldg_amd.LDG(p, 11, 4, 3, precision=precision)      # 132 elements: no multiple of 5, 7, 8, 14, 16 or 32
    u = _noisy(g, p)
    ref = _answers(lib, g, u, 0, 0)
    for c in range(1, lib.ldg_test_candidates()):
        for grad, rhs in ((c, 0), (0, c), (c, c)):
            print(f"candidates p={p} precision={precision} grad {grad} rhs {rhs}", flush=True)
            k, state, ke = _answers(lib, g, u, grad, rhs)
            assert np.array_equal(k, ref[0]) and np.array_equal(state, ref[1])
            assert np.allclose(ke, ref[2], rtol=1e-13, atol=0)
    g.close()


@pytest.mark.parametrize("precision", PRECISIONS)
@pytest.mark.parametrize("per_step", [False, True])
def test_candidates_add_the_same_corrections(per_step, precision):
    """The gate bound lies at the median of the corrections' RMS, so that it
    is open in some elements and closed in others."""
    lib = _candidates()
    g = ldg_amd.LDG(2, 11, 4, 3, precision=precision)
    u = _noisy(g, 9)
    c = C.Closure(2, 256, 0, seed=4)
    rng = np.random.default_rng(3)
    norm = np.concatenate([np.zeros(c.nin), rng.uniform(0.5, 2.0, c.nin), rng.standard_normal(c.nout),
                           rng.uniform(0.5, 2.0, c.nout)]).astype(np.float32)
    c.set(norm=norm)
    lib.ldg_test_set_candidates(g._h, 0, 0)
    plain = g.rhs(u)
    C.attach(g, c, 1e30, per_step=per_step)
    y = (g.rhs(u) - plain).reshape(g.K, -1)
    rms = np.sqrt(np.mean(((y - norm[2 * c.nin:2 * c.nin + c.nout]) / norm[2 * c.nin + c.nout:]) ** 2, axis=1))
    C.attach(g, c, float(np.median(rms)), per_step=per_step)
    ref = _answers(lib, g, u, 0, 0)
    off, total = C.gated(g)
    assert 0 < off < total
    assert not np.array_equal(ref[0], plain)
    for cand in range(1, lib.ldg_test_candidates()):
        print(f"closure, candidate {cand} precision={precision} per_step={per_step}", flush=True)
        k, state, ke = _answers(lib, g, u, cand, cand)
        assert C.gated(g) == (off, total)
        assert np.array_equal(k, ref[0]) and np.array_equal(state, ref[1])
        assert np.allclose(ke, ref[2], rtol=1e-13, atol=0)
    g.close()
    c.close()


# just above the element counts up to which small-mesh kernels run in the mixed path
@pytest.mark.parametrize("p,mesh", [(1, (31, 31, 31)), (2, (24, 24, 23)), (3, (20, 19, 20)), (4, (16, 16, 15)),
                                    (5, (13, 13, 11))])
def test_noalloc_equals_ldg_rhs_above_the_small_meshes(p, mesh):
    print(f"ldg_rhs_noalloc mixed p={p} {mesh}", flush=True)
    hip = _hip()
    g = ldg_amd.LDG(p, *mesh, precision=ldg_amd.LDG_MIXED)
    u = _noisy(g, p)
    assert np.array_equal(_noalloc_rhs(hip, g.cfg, u), g.rhs(u))
    g.close()
