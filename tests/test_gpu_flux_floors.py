"""The Euler fluxes under density and pressure floors against the oracle, with
cells below the floors: Apollo floors the conserved and the primitive state
before it forms the sound speeds and the Roe averages (wxeulereqn.cc:1324-1341)."""
import numpy as np
import pytest

from apollo_amd import engine as E
from oracle import oracle as O

from cases import Case, euler_case, fp64_parity, rounding_floor

pytestmark = pytest.mark.gpu


def _case(N, m, flux):
    base = euler_case(n=6, N=N, m=m, flux=flux)
    p = base.params
    return Case(base.mesh, E.Params(N, p.eqn, flux=flux, gas_gamma=1.4, min_density=1e-2,
                                    min_pressure=1e-3), "euler with floors")


def _check(case, q):
    eng = E.Engine(case.mesh, case.params)
    out = np.zeros_like(q)
    dt = eng.rhs(0.0, q, out, cfl=0.5)
    eng.close()
    fp64_parity(case, out, q, floor=rounding_floor(case, q))
    _, speed = case.oracle_rhs(q)
    ref = O.suggested_dt(case.omesh, 0.5, speed)
    assert abs(dt - ref) <= 1e-12 * ref


@pytest.mark.parametrize("flux", [E.FLUX_HLL, E.FLUX_ROE])
@pytest.mark.parametrize("N,m", [(1, 5), (2, 4), (4, 4), (5, 5)])
def test_riemann_flux_of_cells_below_the_floors(flux, N, m):
    case = _case(N, m, flux)
    # pressure: two cells that share a face, one alone, both signs of their velocity
    q = case.state(amp=1e-3)
    for k, u, e in ((6, 1.0, 0.45), (7, 0.7, 0.1), (30, -0.5, 0.1)):
        q[k] = 0.0
        q[k, :, 0], q[k, :, 1], q[k, :, -1] = 1.0, u, e
    _check(case, q)
    # density
    q = case.state(amp=1e-3)
    q[7] = 0.0
    q[7, :, 0], q[7, :, 1], q[7, :, -1] = -0.1, 0.01, 2.0
    _check(case, q)


@pytest.mark.parametrize("flux", [E.FLUX_LF, E.FLUX_HLL, E.FLUX_ROE])
def test_states_above_the_floors_do_not_see_them(flux):
    case = _case(3, 4, flux)
    q = case.state(amp=1e-3)
    with_floors, without = np.zeros_like(q), np.zeros_like(q)
    for params, out in ((case.params, with_floors),
                        (E.Params(3, case.params.eqn, flux=flux, gas_gamma=1.4), without)):
        eng = E.Engine(case.mesh, params)
        eng.rhs(0.0, q, out)
        eng.close()
    assert np.array_equal(with_floors, without)
