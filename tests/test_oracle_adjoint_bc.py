"""The oracle's discrete adjoint at the Euler boundaries: walls, inflow,
Dirichlet states and zero gradient, against central differences of its RHS."""
import pytest

from oracle import oracle as O

from adjoint_bc import KINDS, boundary_case, check_dot_product, subsonic_state
from cases import to_oracle


@pytest.mark.parametrize("kinds", KINDS)
@pytest.mark.parametrize("N,m", [(2, 5), (3, 4)])
def test_oracle_adjoint_at_euler_boundaries(N, m, kinds):
    case = boundary_case(N, m, kinds)
    check_dot_product(to_oracle(case.params.eqn, subsonic_state(case)),
                      lambda q: O.rhs(case.omesh, case.ophys, 0.0, q)[0],
                      lambda q, w: O.adjoint_rhs(case.omesh, case.ophys, 0.0, q, w),
                      zero=3 if m == 4 else None)
