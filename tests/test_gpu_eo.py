"""The even-odd cubature kernel (FP64, N <= 4) against the oracle where its
groups of 32 elements and its group widths change: fewer elements than a
group, an exact group and one more, meshes on either side of the limit of the
eight-wave groups (256 groups) and in the range of the one-wave groups, with
a partial last group; every epilogue (RHS, LSERK4 stage, SSP combination);
element-pair variables of even and odd number."""
import numpy as np
import pytest

from apollo_amd import engine as E
from oracle import oracle as O

from cases import (Case, euler_case, ffs_case, ffs_state, fp64_parity, from_oracle, maxwell_case,
                   rel_l2, rounding_floor, to_oracle)

pytestmark = pytest.mark.gpu


def _engine(case, algorithm=E.ALGO_CUBATURE):
    p = case.params
    return E.Engine(case.mesh, E.Params(p.order, p.eqn, flux=p.flux, gas_gamma=p.gas_gamma, c0=p.c0,
                                        chi=p.chi, gamma_ph=p.gamma_ph, bcs=p.bcs, algorithm=algorithm))


def _check(case, q, t=0.0):
    eng = _engine(case)
    out = np.zeros_like(q)
    dt = eng.rhs(t, q, out, cfl=0.5)
    eng.close()
    fp64_parity(case, out, q, t, floor=rounding_floor(case, q, t))
    _, speed = case.oracle_rhs(q, t)
    ref = O.suggested_dt(case.omesh, 0.5, speed)
    assert abs(dt - ref) <= 1e-13 * ref


# K = 18 (one partial group), 32 (exactly one), 50; 8192 and 8450 lie on
# either side of 256 groups
@pytest.mark.parametrize("n", [3, 4, 5, 64, 65])
@pytest.mark.parametrize("N,m", [(1, 5), (2, 4), (3, 5), (4, 4), (4, 5)])
def test_eo_sizes(n, N, m):
    case = euler_case(n=n, N=N, m=m)
    _check(case, case.state(amp=1e-3))


@pytest.mark.parametrize("N,m", [(3, 5), (4, 4)])
def test_eo_one_wave_groups(N, m):
    """K = 132098: 4129 groups, one wave each, the last one partial."""
    case = euler_case(n=257, N=N, m=m)
    _check(case, case.state(amp=1e-3))


@pytest.mark.parametrize("N", [1, 2, 3, 4])
def test_eo_boundaries(N):
    """Inflow, walls, outflow; the time-dependent vortex boundary; PEC and TM
    walls of both Maxwell systems in the cubature form."""
    for flux in (E.FLUX_LF, E.FLUX_HLL):
        case = ffs_case(N=N, m=5, flux=flux, limiter=False)
        _check(case, ffs_state(case, "smooth", seed=N))
    case = euler_case(n=7, N=N, m=4, periodic=False)
    _check(case, case.state(amp=1e-3), 0.37)
    for m, bc, flux in ((3, E.BC_PEC, E.FLUX_UPWIND), (8, E.BC_MAXWELL_TM, E.FLUX_LF)):
        case = maxwell_case(n=6, N=N, m=m, bc=bc, flux=flux)
        _check(case, case.state())


@pytest.mark.parametrize("n", [3, 4, 65])
@pytest.mark.parametrize("N", [3, 4])
def test_eo_eight_variables(N, n):
    """The last order of the 8-variable system on this kernel and the first
    that the MFMA kernel takes (the same bits as when it is asked for)."""
    case = maxwell_case(n=n, N=N, m=8, bc=E.BC_PEC)
    q = case.state()
    _check(case, q)
    out = [np.zeros_like(q), np.zeros_like(q)]
    for o, algorithm in zip(out, (E.ALGO_CUBATURE, E.ALGO_CUBATURE_MFMA)):
        eng = _engine(case, algorithm)
        eng.rhs(0.0, q, o)
        eng.close()
    assert np.array_equal(out[0], out[1]) == (N == 4)


@pytest.mark.parametrize("N,m,n", [(1, 4, 156), (1, 4, 157), (2, 5, 157), (1, 8, 128), (2, 8, 157)])
def test_eo_one_wave_groups_small_orders(N, m, n):
    """One-wave groups from 1536 groups on (K = 49152; n = 156 and 157 lie on
    either side), for eight variables at N = 1 from 1024 on."""
    if m == 8:
        case = maxwell_case(n=n, N=N, m=m, bc=E.BC_PEC)
        _check(case, case.state())
    else:
        case = euler_case(n=n, N=N, m=m)
        _check(case, case.state(amp=1e-3))


@pytest.mark.parametrize("flux", [E.FLUX_UPWIND, E.FLUX_LF])
@pytest.mark.parametrize("N,n", [(1, 128), (1, 129), (1, 157), (2, 129)])
def test_eo_tm_meshes(N, n, flux):
    """TM meshes at the limits of the vector-ALU kernel's FP64 form, between
    K = 32768 (the last four-wave mesh here) and, at N = 1, 49152 (one-wave
    groups from there); PEC walls, a partial last group but for n = 128."""
    case = maxwell_case(n=n, N=N, m=3, bc=E.BC_PEC, flux=flux)
    q = case.state()
    _check(case, q)
    eng = _engine(case)
    got = q.copy()
    eng.lserk4(0.0, 1e-4, 1, got)
    eng.close()
    with O.exact_geometry():
        ref = from_oracle(case.params.eqn, O.lserk4(case.omesh, case.ophys, 0.0, 1e-4, 1,
                                                    to_oracle(case.params.eqn, q)))
    assert rel_l2(got - q, ref - q) <= 1e-11


@pytest.mark.parametrize("N,n", [(2, 5), (3, 65), (4, 20)])
def test_eo_steppers(N, n):
    case = euler_case(n=n, N=N, m=4)
    q0 = case.state(amp=1e-3)
    eng = _engine(case)
    q = q0.copy()
    eng.lserk4(0.0, 1e-3, 3, q)
    cfl = 0.5 / (2 * N + 1)
    qs = q0.copy()
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


@pytest.mark.parametrize("N", [1, 4])
def test_eo_reports_bad_states(N):
    """A negative density, a negative pressure and a NaN at one interior node."""
    case = euler_case(n=6, N=N, m=5)
    for var, value, status in ((0, -1.0, 8), (4, 0.0, 9), (2, np.nan, 9)):
        q = case.state(amp=1e-3)
        q[7, :, var] = value
        eng = _engine(case)
        with pytest.raises(E.ApolloError) as e:
            eng.rhs(0.0, q, np.zeros_like(q))
        eng.close()
        assert e.value.status == status


@pytest.mark.parametrize("n", [3, 4, 5, 40])
@pytest.mark.parametrize("N,m", [(1, 4), (2, 5), (3, 5), (4, 4), (4, 3), (2, 8)])
def test_eo_adjoint_sizes(n, N, m):
    """The transposed RHS on a partial, an exact and several groups (eight
    waves each), periodic (Euler) or with reflecting walls (Maxwell)."""
    case = euler_case(n=n, N=N, m=m) if m in (4, 5) else maxwell_case(n=n, N=N, m=m, bc=E.BC_PEC)
    _check_adjoint(case)


@pytest.mark.parametrize("N,m,n,periodic", [(3, 4, 65, True), (4, 4, 182, True), (2, 4, 20, False),
                                            (2, 4, 257, True)])
def test_eo_adjoint_groups(N, m, n, periodic):
    """Four-wave groups (n = 65, and the vortex boundary's), one-wave groups
    where four-wave ones fill a CU's LDS (n = 182, 2071 groups) and where
    they do not (n = 257, 4129 groups of four waves)."""
    _check_adjoint(euler_case(n=n, N=N, m=m, periodic=periodic))


def _check_adjoint(case):
    q = case.state(amp=1e-3)
    lam = np.random.default_rng(5).standard_normal(q.shape)
    eng = E.Engine(case.mesh, case.params)
    out = np.zeros_like(q)
    eng.adjoint_rhs(0.3, q, lam, out)
    eng.close()
    with O.exact_geometry():
        ref = from_oracle(case.params.eqn, O.adjoint_rhs(case.omesh, case.ophys, 0.3,
                                                         to_oracle(case.params.eqn, q),
                                                         to_oracle(case.params.eqn, lam)))
    assert rel_l2(out, ref) <= 1e-12


def test_eo_reverse_lserk4_partial_groups():
    """Reverse stages whose next-stage weights cross a partial last group."""
    case = euler_case(n=9, N=2, m=5, periodic=False)
    q0 = case.state(amp=1e-3)
    gT = np.random.default_rng(2).standard_normal(q0.shape)
    eng = E.Engine(case.mesh, case.params)
    g0, qT = np.zeros_like(q0), np.zeros_like(q0)
    eng.lserk4_adjoint(0.2, 0.01, 3, 2, q0, gT, g0, qT)
    eng.close()
    with O.exact_geometry():
        ref = from_oracle(case.params.eqn, O.lserk4_adjoint(case.omesh, case.ophys, 0.2, 0.01, 3,
                                                            to_oracle(case.params.eqn, q0),
                                                            to_oracle(case.params.eqn, gT)))
    assert rel_l2(g0, ref) <= 1e-11
