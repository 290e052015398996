"""Kinetic energies at p = 5 do not depend on which kernels ran: an instance
of an ensemble whose elements together are past the small meshes records the
energies it records alone, bit by bit (its kernels take 3 elements to a
workgroup there, 1 alone), and so does a handle under every candidate."""
import numpy as np
import pytest

import ldg_amd
from test_gpu_candidates import _answers, _candidates, _noisy

pytestmark = pytest.mark.gpu


# 2 x 7 x 8 x 9 = 1008 elements > 900 (FP64), 3 x 9 x 9 x 8 = 1944 > 1800 (mixed)
@pytest.mark.parametrize("precision,count,mesh", [(ldg_amd.LDG_FP64, 2, (7, 8, 9)), (ldg_amd.LDG_MIXED, 3, (9, 9, 8))])
@pytest.mark.parametrize("graph", [False, True])
def test_instance_energy_is_the_single_solvers(precision, count, mesh, graph):
    print(f"p=5 ensemble of {count} x {mesh}, precision={precision} graph={graph}", flush=True)
    members = [{"p": 5, "nx": mesh[0], "ny": mesh[1], "nz": mesh[2], "Re": 900.0 + 300 * i, "M0": 0.1, "V0": 1.0 + 0.02 * i,
                "phase": (0.3 * i, 1.1, 2.0)} for i in range(count)]
    ens = ldg_amd.Ensemble(members, precision=precision)
    ens.initial_condition()
    ens.set_graph(graph)
    dts = ens.time_steps(0.01)
    u0 = [ens.get_instance_state(i) for i in range(count)]
    ke = ens.step(dts, 5)
    for i, d in enumerate(members):
        g = ldg_amd.LDG(5, *mesh, Re=d["Re"], M0=d["M0"], V0=d["V0"], precision=precision)
        g.set_state(u0[i])
        np.testing.assert_array_equal(ke[:, i], g.step(dts[i], 5), err_msg=f"instance {i}")
        np.testing.assert_array_equal(ens.get_instance_state(i), g.get_state(), err_msg=f"instance {i}")
        g.close()
    ens.close()


@pytest.mark.parametrize("precision", [ldg_amd.LDG_FP64, ldg_amd.LDG_MIXED])
def test_candidates_record_the_same_energies(precision):
    lib = _candidates()
    g = ldg_amd.LDG(5, 11, 4, 3, precision=precision)
    u = _noisy(g, 5)
    energies = [_answers(lib, g, u, 0, c)[2] for c in range(lib.ldg_test_candidates())]
    for ke in energies[1:]:
        np.testing.assert_array_equal(ke, energies[0])
    g.close()
