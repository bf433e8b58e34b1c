"""The engine's discrete adjoint at the Euler boundaries: walls, inflow,
Dirichlet states and zero gradient, against central differences of its own RHS
and against the oracle, on both adjoint kernels."""
import numpy as np
import pytest

from apollo_amd import engine as E
from oracle import oracle as O

from adjoint_bc import KINDS, boundary_case, check_dot_product, subsonic_state
from cases import from_oracle, rel_l2, to_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kinds", KINDS)
@pytest.mark.parametrize("N,m", [(1, 5), (3, 4), (4, 5), (5, 4)])
def test_adjoint_at_euler_boundaries(N, m, kinds):
    case = boundary_case(N, m, kinds)
    q = subsonic_state(case)
    eng = E.Engine(case.mesh, case.params)

    def rhs(x):
        out = np.zeros_like(x)
        eng.rhs(0.0, x, out)
        return out

    def adjoint(x, w):
        out = np.zeros_like(x)
        eng.adjoint_rhs(0.0, x, w, out)
        return out

    check_dot_product(q, rhs, adjoint)
    lam = np.random.default_rng(4).standard_normal(q.shape)
    got = adjoint(q, lam)
    eng.close()
    with O.exact_geometry():
        ref = O.adjoint_rhs(case.omesh, case.ophys, 0.0, to_oracle(case.params.eqn, q),
                            to_oracle(case.params.eqn, lam))
    assert rel_l2(got, from_oracle(case.params.eqn, ref)) <= 1e-12
