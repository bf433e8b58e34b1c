"""The even-odd nodal kernel (Maxwell, FP64) against the oracle where its groups
of 16 elements and its group widths change: fewer elements than a group, exact
groups and a partial last one, every order (whole and padded units of two
mirrored pairs), the last mesh of the TM kernel's range and one behind it,
and groups of four, two and one waves of the 8-variable system."""
import numpy as np
import pytest

from apollo_amd import engine as E
from oracle import oracle as O

from cases import fp64_parity, from_oracle, maxwell_case, rel_l2, rounding_floor, to_oracle

pytestmark = pytest.mark.gpu


def _check(case, t=0.0):
    q = case.state(amp=1e-3)
    eng = E.Engine(case.mesh, case.params)
    out = np.zeros_like(q)
    dt = eng.rhs(t, q, out, cfl=0.5)
    eng.close()
    fp64_parity(case, out, q, t, floor=rounding_floor(case, q, t))
    _, speed = case.oracle_rhs(q, t)
    ref = O.suggested_dt(case.omesh, 0.5, speed)
    assert abs(dt - ref) <= 1e-13 * ref


# K = 8, 18, 32, 50
@pytest.mark.parametrize("n", [2, 3, 4, 5])
@pytest.mark.parametrize("N", range(1, 9))
@pytest.mark.parametrize("m", [3, 8])
def test_eo_linear_sizes(n, N, m):
    kw = dict(chi=1.1, gph=0.9) if m == 8 else {}
    _check(maxwell_case(n=n, N=N, m=m, bc=E.BC_PEC if n & 1 else E.BC_MAXWELL_TM,
                        flux=E.FLUX_UPWIND if m == 3 and n & 1 else E.FLUX_LF, **kw))


# 512 groups of 16 and one more (TM; at N = 8 the line is 256); 8-variable:
# 529 groups (two waves each) and 1036 (one wave each at N <= 4)
@pytest.mark.parametrize("n,N,m", [(64, 3, 3), (65, 3, 3), (64, 7, 3), (45, 8, 3), (46, 8, 3),
                                   (64, 4, 8), (65, 4, 8), (65, 6, 8), (91, 1, 8), (91, 4, 8)])
def test_eo_linear_groups(n, N, m):
    _check(maxwell_case(n=n, N=N, m=m, bc=E.BC_PEC, **(dict(chi=1.0, gph=1.0) if m == 8 else {})))


@pytest.mark.parametrize("n", [4, 5])
@pytest.mark.parametrize("N,m", [(2, 3), (5, 3), (1, 8), (4, 8)])
def test_eo_linear_steppers(n, N, m):
    """The LSERK4 stage and the SSP combination on exact and partial groups."""
    case = maxwell_case(n=n, N=N, m=m, bc=E.BC_PEC, **(dict(chi=1.0, gph=1.0) if m == 8 else {}))
    q0 = case.state(amp=1e-3)
    cfl = 0.5 / (2 * N + 1)
    eng = E.Engine(case.mesh, case.params)
    q, qs = q0.copy(), q0.copy()
    eng.lserk4(0.0, 1e-3, 3, q)
    dts = eng.ssp_advance(0.0, 3e-3, 1e-3, cfl, qs)
    eng.close()
    with O.exact_geometry():
        ref = from_oracle(case.params.eqn, O.lserk4(case.omesh, case.ophys, 0.0, 1e-3, 3,
                                                    to_oracle(case.params.eqn, q0)))
        refs, dto = O.ssp_advance(case.omesh, case.ophys, 0.0, 3e-3, 1e-3, cfl,
                                  to_oracle(case.params.eqn, q0))
    assert rel_l2(q - q0, ref - q0) <= 1e-11
    assert len(dts) == len(dto) and np.abs(dts - dto).max() <= 1e-13 * dto.max()
    assert rel_l2(qs - q0, from_oracle(case.params.eqn, refs) - q0) <= 1e-11
