"""The discrete adjoint at states the wave speed does not exist for: a cell
whose sound speed squared is negative is reported (APL_ERR_NAN) at every
order, and one without pressure at rest, whose speed never leads, is not."""
import numpy as np
import pytest

from apollo_amd import engine as E
from oracle import oracle as O

from cases import euler_case, from_oracle, rel_l2, to_oracle

pytestmark = pytest.mark.gpu


def _with_cell(case, rho, u, v, energy):
    q = case.state(amp=1e-3)
    q[7] = 0.0
    q[7, :, 0], q[7, :, 1], q[7, :, 2], q[7, :, -1] = rho, rho * u, rho * v, energy
    return q


# orders of both adjoint kernels: N = 5 and five variables at N = 4 are on MFMA
@pytest.mark.parametrize("N", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("m", [4, 5])
def test_adjoint_reports_inadmissible_cells(N, m):
    case = euler_case(n=6, N=N, m=m)
    eng = E.Engine(case.mesh, case.params)
    # negative pressure on the slower and on the faster side of its faces, a
    # negative density with a positive pressure
    for cell in ((1.0, 0.0, 0.0, -0.05), (1.0, 8.0, 3.0, 36.0), (-1.0, 0.1, 0.1, 2.0)):
        q = _with_cell(case, *cell)
        lam = np.random.default_rng(3).standard_normal(q.shape)
        with pytest.raises(E.ApolloError) as e:
            eng.adjoint_rhs(0.0, q, lam, np.zeros_like(q))
        assert e.value.status == 7
    # the call after a reported one starts clean
    q = case.state(amp=1e-3)
    eng.adjoint_rhs(0.0, q, q.copy(), np.zeros_like(q))
    eng.close()


@pytest.mark.parametrize("N,m", [(1, 4), (2, 5), (3, 4), (4, 4), (5, 4)])
def test_adjoint_of_a_cell_without_pressure_at_rest(N, m):
    case = euler_case(n=6, N=N, m=m)
    q = _with_cell(case, 1.0, 0.0, 0.0, 0.0)
    lam = np.random.default_rng(3).standard_normal(q.shape)
    out = np.zeros_like(q)
    eng = E.Engine(case.mesh, case.params)
    eng.adjoint_rhs(0.0, q, lam, out)
    eng.close()
    with O.exact_geometry():
        ref = from_oracle(case.params.eqn, O.adjoint_rhs(case.omesh, case.ophys, 0.0,
                                                         to_oracle(case.params.eqn, q),
                                                         to_oracle(case.params.eqn, lam)))
    assert np.isfinite(ref).all()
    assert rel_l2(out, ref) <= 1e-12
