"""The steppers on the wide meshes' instantiations of the even-odd kernels, each
with a partial last group: one- and two-wave groups in the LSERK4 stage, the
SSP combination and the reverse stage (whose next weights pass between the
lanes of a single wave)."""
import numpy as np
import pytest

from apollo_amd import engine as E
from oracle import oracle as O

from cases import euler_case, from_oracle, maxwell_case, rel_l2, to_oracle

pytestmark = pytest.mark.gpu


def _steppers(case, dt):
    q0 = case.state(amp=1e-3)
    eqn, cfl = case.params.eqn, 0.5 / (2 * case.params.order + 1)
    eng = E.Engine(case.mesh, case.params)
    q, qs = q0.copy(), q0.copy()
    eng.lserk4(0.0, dt, 1, q)
    dts = eng.ssp_advance(0.0, 1.5 * dt, dt, cfl, qs)
    eng.close()
    with O.exact_geometry():
        ref = from_oracle(eqn, O.lserk4(case.omesh, case.ophys, 0.0, dt, 1, to_oracle(eqn, q0)))
        refs, dto = O.ssp_advance(case.omesh, case.ophys, 0.0, 1.5 * dt, dt, cfl, to_oracle(eqn, q0))
    assert rel_l2(q - q0, ref - q0) <= 1e-11
    assert len(dts) == len(dto) and np.abs(dts - dto).max() <= 1e-13 * dto.max()
    assert rel_l2(qs - q0, from_oracle(eqn, refs) - q0) <= 1e-11


# 8 variables, N = 4: 529 groups of 16 elements (two waves each), 1036 (one)
@pytest.mark.parametrize("n", [65, 91])
def test_nodal_steppers(n):
    _steppers(maxwell_case(n=n, N=4, m=8, bc=E.BC_PEC, chi=1.0, gph=1.0), 1e-4)


# groups of 32 elements: 6163 (the line is 6144 at N = 1, 2), 4129 (4096 at
# N = 3 and four variables at N = 4), 1041 (1024 for five at N = 4), one wave each
@pytest.mark.parametrize("N,m,n", [(1, 5, 314), (2, 4, 314), (3, 5, 257), (4, 4, 257), (4, 5, 129)])
def test_cubature_steppers(N, m, n):
    _steppers(euler_case(n=n, N=N, m=m), 1e-4)


# 1041 groups: one wave each for four variables at N = 4 and five at N = 3
@pytest.mark.parametrize("N,m", [(4, 4), (3, 5)])
def test_reverse_lserk4(N, m):
    case = euler_case(n=129, N=N, m=m)
    eqn = case.params.eqn
    q0 = case.state(amp=1e-3)
    gT = np.random.default_rng(2).standard_normal(q0.shape)
    g0, qT = np.zeros_like(q0), np.zeros_like(q0)
    eng = E.Engine(case.mesh, case.params)
    eng.lserk4_adjoint(0.0, 1e-3, 2, 1, q0, gT, g0, qT)
    eng.close()
    with O.exact_geometry():
        ref = O.lserk4_adjoint(case.omesh, case.ophys, 0.0, 1e-3, 2, to_oracle(eqn, q0), to_oracle(eqn, gT))
    assert rel_l2(g0, from_oracle(eqn, ref)) <= 1e-11
