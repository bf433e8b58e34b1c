"""Rounding of the even-odd kernels: their distance from the RHS in long
double, from the same tables, is that of the MFMA kernels on the same state.

Both sum the same products; the even-odd form adds one rounding to form the
even and odd parts and one to recombine them, and sums half-length rows of
twice the size, so its error may be a factor sqrt(2) larger where rounding
is all there is.  The nearly constant states of a fine mesh make the rest
visible: the volume and surface terms, of order |F| / h each, cancel, and an
asymmetry of the setup's tables in the last digits does not."""
import numpy as np
import pytest

from apollo_amd import engine as E

from cases import Case

pytestmark = pytest.mark.gpu
LD = np.longdouble


def _case(N, eqn, flux):
    """A periodic square as fine as a 100 x 100 mesh of a unit domain."""
    mesh = E.structured_mesh(8, 0.0, 0.08, 0.0, 0.08, 0.1, 5, True)
    ph = {"chi": 1.0, "gamma_ph": 1.0} if eqn == E.EQN_PHMAXWELL8 else {}
    return mesh, lambda algorithm: E.Params(N, eqn, flux=flux, algorithm=algorithm, gas_gamma=1.4, **ph)


def _state(case, m, euler, seed):
    """A smooth state, continuous across the faces: modes of the domain around values of order 1."""
    g = np.random.default_rng(seed)
    x, y = case.omesh.x, case.omesh.y
    w = []
    for _ in range(m):
        k = 2 * np.pi / 0.08 * g.integers(1, 3, 2)
        w.append(0.02 * np.sin(k[0] * x + g.uniform(0, 6)) * np.cos(k[1] * y + g.uniform(0, 6)) + g.uniform(0.5, 1.0))
    if not euler:
        return np.ascontiguousarray(np.stack(w, -1))
    rho, u, v, p = w[0], w[1] - 0.4, w[2] - 0.9, w[3]
    c = [rho, rho * u, rho * v] + ([0.1 * rho] if m == 5 else [])
    return np.ascontiguousarray(np.stack(c + [p / 0.4 + 0.5 * rho * (u * u + v * v + (0.01 if m == 5 else 0.0))], -1))


def _flux(eqn, q):
    """F, G and the wave speed in long double (c0 = 1; chi = gamma = 1 for 8 variables)."""
    if eqn == E.EQN_MAXWELL_TM3:
        a, b, h = np.moveaxis(q, -1, 0)
        z = 0 * a
        return np.stack([-h, z, -a], -1), np.stack([b, a, z], -1), 1 + z
    if eqn == E.EQN_PHMAXWELL8:
        ex, ey, ez, bx, by, bz, ph, ps = np.moveaxis(q, -1, 0)
        return (np.stack([ph, bz, -by, ps, -ez, ey, ex, bx], -1),
                np.stack([-bz, ph, bx, ez, ps, -ex, ey, by], -1), 1 + 0 * ex)
    rho, mu, mv, e = q[..., 0], q[..., 1], q[..., 2], q[..., -1]
    u, v = mu / rho, mv / rho
    w = q[..., 3] / rho if q.shape[-1] == 5 else 0 * u
    gam = LD(1.4)
    k2 = u * u + v * v + w * w
    p = (gam - 1) * (e - rho * k2 / 2)
    mid = [rho * w * u] if q.shape[-1] == 5 else []
    mid2 = [rho * w * v] if q.shape[-1] == 5 else []
    return (np.stack([mu, mu * u + p, mu * v] + mid + [(e + p) * u], -1),
            np.stack([mv, mv * u, mv * v + p] + mid2 + [(e + p) * v], -1), np.sqrt(k2) + np.sqrt(gam * p / rho))


def _rhs(N, eqn, mesh, geom, q):
    """The LF RHS in long double from the stored operators and geometry."""
    op = lambda k: E.host_operator(N, k).astype(LD)  # noqa: E731
    w, gw, r = op(5), op(7), op(8)
    Np, Nc, Ng = r.size, w.size, gw.size
    V, Dr, Ds = (op(k).reshape(Nc, Np) for k in (0, 1, 2))
    If, VVT = op(3).reshape(3 * Ng, Np), op(4).reshape(Np, Np)
    Ar, As, L = (VVT @ Dr.T) * w, (VVT @ Ds.T) * w, (VVT @ If.T) * np.tile(gw, 3)
    # the metric factors as the engine stores them: J times the gradients, in 64 bits
    jrx, jsx, jry, jsy = ((geom[:, 4] * geom[:, k]).astype(LD)[:, None, None] for k in range(4))
    q, geom = q.astype(LD), geom.astype(LD)
    J = geom[:, 4, None, None]
    mul = lambda A, x: np.einsum("ij,kjm->kim", A, x)  # noqa: E731
    F, G, _ = _flux(eqn, mul(V, q))
    out = mul(Ar, jrx * F + jry * G) + mul(As, jsx * F + jsy * G)
    tr = mul(If, q).reshape(mesh.K, 3, Ng, -1)
    et = E.host_connectivity(mesh).reshape(mesh.K, 3, 2)
    qP = tr[et[:, :, 0], et[:, :, 1]][:, :, ::-1]
    n = geom[:, 5:].reshape(mesh.K, 3, 3)
    nx, ny, sj = (n[:, :, k, None, None] for k in range(3))
    FM, GM, cM = _flux(eqn, tr)
    FP, GP, cP = _flux(eqn, qP)
    f = sj * (nx * (FM + FP) + ny * (GM + GP) + np.maximum(cM, cP)[..., None] * (tr - qP)) / 2
    return (out - mul(L, f.reshape(mesh.K, 3 * Ng, -1))) / J


def _errors(N, eqn, algorithms):
    mesh, params = _case(N, eqn, E.FLUX_LF)
    case = Case(mesh, params(E.ALGO_AUTO))
    total = np.zeros(len(algorithms))
    for seed in range(3):
        q = _state(case, params(E.ALGO_AUTO).m, eqn in (E.EQN_EULER4, E.EQN_EULER5), seed)
        ref = None
        for i, alg in enumerate(algorithms):
            eng = E.Engine(mesh, params(alg))
            if ref is None:
                ref = _rhs(N, eqn, mesh, eng.geometry()[0].reshape(mesh.K, 14), q)
            out = np.zeros_like(q)
            eng.rhs(0.0, q, out)
            eng.close()
            d = (out - ref).astype(np.float64)
            total[i] += np.sum(d * d) / float(np.sum(ref * ref))
    return np.sqrt(total / 3)


@pytest.mark.parametrize("N", range(1, 9))
@pytest.mark.parametrize("eqn", [E.EQN_MAXWELL_TM3, E.EQN_PHMAXWELL8])
def test_eo_nodal_rounding(N, eqn):
    here, mfma = _errors(N, eqn, (E.ALGO_AUTO, E.ALGO_NODAL_MFMA))
    print("N %d: even-odd %.2e, MFMA %.2e, ratio %.2f" % (N, here, mfma, here / mfma))
    assert here <= np.sqrt(2.0) * mfma


@pytest.mark.parametrize("N", range(1, 5))
@pytest.mark.parametrize("eqn", [E.EQN_EULER4, E.EQN_EULER5])
def test_eo_cubature_rounding(N, eqn):
    here, mfma = _errors(N, eqn, (E.ALGO_CUBATURE, E.ALGO_CUBATURE_MFMA))
    print("N %d: even-odd %.2e, MFMA %.2e, ratio %.2f" % (N, here, mfma, here / mfma))
    assert here <= np.sqrt(2.0) * mfma


def _adjoint(N, mesh, geom, lam):
    """J^T lam of the TM system with the LF flux, in long double from the stored operators and geometry."""
    op = lambda k: E.host_operator(N, k).astype(LD)  # noqa: E731
    w, gw, Np = op(5), op(7), op(8).size
    Nc, Ng = w.size, gw.size
    V, Dr, Ds = (op(k).reshape(Nc, Np) for k in (0, 1, 2))
    If, VVT = op(3).reshape(3 * Ng, Np), op(4).reshape(Np, Np)
    F, G, _ = _flux(E.EQN_MAXWELL_TM3, np.eye(3).astype(LD))     # rows: the fluxes of the unit states
    t = lambda A, x: np.einsum("ij,kim->kjm", A, x)  # noqa: E731
    jrx, jsx, jry, jsy = ((geom[:, 4] * geom[:, k]).astype(LD)[:, None, None] for k in range(4))
    lh = lam.astype(LD) / geom[:, 4].astype(LD)[:, None, None]
    pr, ps = t((VVT @ Dr.T) * w, lh), t((VVT @ Ds.T) * w, lh)
    out = t(V, (jrx * pr + jsx * ps) @ F.T + (jry * pr + jsy * ps) @ G.T)
    n = geom[:, 5:].reshape(mesh.K, 3, 1, 3).astype(LD)
    S = -n[..., 2:] * t((VVT @ If.T) * np.tile(gw, 3), lh).reshape(mesh.K, 3, Ng, 3)
    et = E.host_connectivity(mesh).reshape(mesh.K, 3, 2)
    half = (S - S[et[:, :, 0], et[:, :, 1]][:, :, ::-1]) / 2
    f = n[..., :1] * (half @ F.T) + n[..., 1:2] * (half @ G.T) + half
    return out + t(If, f.reshape(mesh.K, 3 * Ng, 3))


def test_eo_adjoint_rounding():
    """The adjoint of weights M mu with smooth mu, whose terms cancel as the
    forward RHS's do, more so with the order: the even-odd kernels (N <= 4) are
    no farther from the long double value than the MFMA kernel at N = 5."""
    err = {}
    for N in range(1, 6):
        mesh, params = _case(N, E.EQN_MAXWELL_TM3, E.FLUX_LF)
        case = Case(mesh, params(E.ALGO_AUTO))
        eng = E.Engine(mesh, case.params)
        geom = eng.geometry()[0].reshape(mesh.K, 14)
        mass = np.linalg.inv(E.host_operator(N, 4).reshape(case.ops.Np, case.ops.Np))
        total = 0.0
        for seed in range(3):
            q = _state(case, 3, False, seed)
            lam = np.ascontiguousarray(geom[:, 4, None, None] * np.einsum("ij,kjm->kim", mass, q))
            out = np.zeros_like(q)
            eng.adjoint_rhs(0.0, q, lam, out)
            ref = _adjoint(N, mesh, geom, lam)
            d = (out - ref).astype(np.float64)
            total += np.sum(d * d) / float(np.sum(ref * ref)) / 3
        eng.close()
        err[N] = np.sqrt(total)
    print(" ".join("N %d: %.2e" % kv for kv in err.items()))
    assert all(err[N] <= err[5] for N in range(1, 5))
