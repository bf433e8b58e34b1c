"""The disc objective and its gradient against the oracle where its 64-element
waves change: a partial only wave, whole waves with a partial last one, waves
off the disc (their gradient block is zeros), a disc that holds everything
and one that holds nothing; the element count is odd against 64 in all."""
import numpy as np
import pytest

from apollo_amd import engine as E
from oracle import oracle as O

from cases import euler_case, from_oracle, maxwell_case, rel_l2, to_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,m,n", [(1, 5, 3), (3, 4, 20), (5, 3, 9), (8, 4, 7)])
@pytest.mark.parametrize("radius", [0.37, 1.5, 50.0, 0.0])
def test_objective_waves(N, m, n, radius):
    case = euler_case(n=n, N=N, m=m) if m != 3 else maxwell_case(n=n, N=N, m=m)
    q = case.state(amp=1e-3)
    var = m - 1
    eng = E.Engine(case.mesh, case.params)
    g = np.full_like(q, 7.0)
    J = eng.objective_disc_sq(q, var, 0.3, -0.2, radius, g)
    J2 = eng.objective_disc_sq(q, var, 0.3, -0.2, radius)
    eng.close()
    qo = to_oracle(case.params.eqn, q)
    vo = int(np.nonzero(to_oracle(case.params.eqn, np.eye(m)[var][None, None])[0, 0])[0][0])
    Jr, gr = O.objective_disc_sq(case.omesh, qo, vo, 0.3, -0.2, radius, qo.shape[-1])
    gr = from_oracle(case.params.eqn, gr)
    assert J == J2
    if radius == 0.0:
        assert J == 0.0 and not g.any()
    else:
        assert abs(J - Jr) <= 1e-13 * abs(Jr) and rel_l2(g, gr) <= 1e-13
