"""The diagnostics of a state that has no right-hand side are refused
(LDG_ENONFINITE), also where its kinetic energy and enstrophy alone would be
finite: a NaN or infinite energy, a density below zero in one element, a
sound speed that is none.  The oracle is the right-hand side itself: refused
exactly when the rate of density or momentum is not finite somewhere."""
import numpy as np
import pytest

import ldg_amd

pytestmark = pytest.mark.gpu


def _put(s, value, node=slice(None)):
    def plant(u):
        u[7, s, node] = value
    return plant


PLANTED = {"plain": lambda u: None, "density nan": _put(0, np.nan, 3), "density below zero": _put(0, -1.0),
           "momentum inf": _put(2, np.inf, 0), "energy nan": _put(4, np.nan, 3), "energy inf": _put(4, np.inf, 5),
           "energy -inf": _put(4, -np.inf, 0), "energy far below zero": _put(4, -2000.0),
           "energy low at a node": _put(4, 100.0, 2)}
REFUSED = set(PLANTED) - {"plain", "energy low at a node"}


@pytest.mark.parametrize("precision", [ldg_amd.LDG_FP64, ldg_amd.LDG_MIXED])
@pytest.mark.parametrize("p", [1, 2, 3, 4, 5])
def test_refused_with_the_right_hand_side(p, precision):
    print(f"diagnostics p={p} precision={precision}", flush=True)
    g = ldg_amd.LDG(p, 3, 4, 3, precision=precision)
    g.initial_condition()
    plain = g.get_state()
    refused = set()
    for name, plant in PLANTED.items():
        u = plain.copy()
        plant(u)
        finite = bool(np.isfinite(g.rhs(u)[:, :4]).all())
        g.set_state(u)
        if finite:
            assert all(np.isfinite(v) for v in g.diagnostics().values()), name
        else:
            with pytest.raises(ldg_amd.LDGError) as e:
                g.diagnostics()
            assert e.value.code == -4, name
            refused.add(name)
    assert refused == REFUSED
    g.set_state(plain)                           # the handle is not left in error
    assert g.diagnostics()["ke_ref"] > 0.1
    g.close()
