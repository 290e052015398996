"""Small meshes run kernels of their own (wave_kernels.hpp; the choice is by
element count, ldg.hip default_cand).  A periodic state on a small mesh and
the same state repeated twice along every axis on a mesh of eight times the
elements (and the same element size) have the same right-hand side element by
element; the counts below put the two on different sides of the choice, and
the kernels agree operation by operation, so the results are equal bit by
bit.  Odd sizes: partial last workgroups on both sides."""
import numpy as np
import pytest

import ldg_amd

pytestmark = pytest.mark.gpu


def _state(g, seed):
    """A smooth state plus noise on every variable."""
    g.initial_condition()
    u = g.get_state()
    rng = np.random.default_rng(seed)
    for s, a in enumerate((1e-3, 2e-2, 2e-2, 2e-2, 1e-1)):
        u[:, s] += a * rng.standard_normal(u[:, s].shape)
    return u


def _repeat(u, mesh):
    nx, ny, nz = mesh
    return np.tile(u.reshape(nz, ny, nx, *u.shape[1:]), (2, 2, 2, 1, 1)).reshape(8 * u.shape[0], *u.shape[1:])


# elements at most 900 (FP64) / 1800 (mixed) workgroups of 16, 7, 4, 2, 1
# elements (p = 1..5), eight times as many above
@pytest.mark.parametrize("precision,p,mesh", [
    (ldg_amd.LDG_FP64, 1, (13, 13, 11)), (ldg_amd.LDG_FP64, 2, (11, 9, 9)), (ldg_amd.LDG_FP64, 3, (9, 8, 7)),
    (ldg_amd.LDG_FP64, 4, (7, 7, 5)), (ldg_amd.LDG_FP64, 5, (5, 5, 5)),
    (ldg_amd.LDG_MIXED, 1, (17, 16, 15)), (ldg_amd.LDG_MIXED, 2, (13, 12, 11)), (ldg_amd.LDG_MIXED, 3, (11, 10, 9)),
    (ldg_amd.LDG_MIXED, 4, (9, 8, 7)), (ldg_amd.LDG_MIXED, 5, (7, 6, 6))])
def test_small_mesh_kernels_are_bitwise_the_others(precision, p, mesh):
    print(f"small mesh p={p} {mesh} precision={precision}", flush=True)
    h = 0.25                                     # element sizes exact in both meshes
    small = ldg_amd.LDG(p, *mesh, xmin=[0.0] * 3, xmax=[n * h for n in mesh], precision=precision)
    large = ldg_amd.LDG(p, *(2 * n for n in mesh), xmin=[0.0] * 3, xmax=[2 * n * h for n in mesh], precision=precision)
    u = _state(small, p)
    ul = _repeat(u, mesh)
    assert np.array_equal(large.rhs(ul), _repeat(small.rhs(u), mesh))
    small.set_state(u)
    large.set_state(ul)
    dt = 1e-4
    ks, kl = small.step(dt, 3), large.step(dt, 3)
    assert np.array_equal(large.get_state(), _repeat(small.get_state(), mesh))
    # same sums (eight times as many terms) in another order
    assert np.allclose(kl, 8 * ks, rtol=1e-13, atol=0)
    small.close()
    large.close()
