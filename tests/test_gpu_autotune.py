"""What the autotuner reports tells the kernels apart: at most orders the
small-mesh kernels take as many elements to a workgroup as the default ones
(7 at p = 2), and are reported negative.  On 8^3 elements they take about two
thirds of the others' time; at p = 4 they fall behind from 13^3 elements on."""
import pytest

import ldg_amd

pytestmark = pytest.mark.gpu

# the candidates of (gradient, right-hand side) per order
CANDIDATES = {2: ({7, 14, -7}, {7, 14, -7}), 4: ({5, 2, -2}, {2, 5, -2})}


@pytest.mark.parametrize("p,nx,small", [(2, 8, True), (4, 32, False)])
def test_reported_candidates_name_the_kernels(p, nx, small):
    g = ldg_amd.LDG(p, nx)
    g.initial_condition()
    (order, grad, rhs), = g.autotune()
    print("autotune", nx, p, grad, rhs, flush=True)
    assert order == p and grad in CANDIDATES[p][0] and rhs in CANDIDATES[p][1]
    assert (grad < 0, rhs < 0) == (small, small)
    g.close()
