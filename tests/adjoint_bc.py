"""A mesh with four different Euler boundaries and the check of an adjoint RHS
against central differences of the forward RHS; used on the engine and on the
oracle."""
import numpy as np

from apollo_amd import engine as E

from cases import Case

GAMMA = 1.4


def boundary_case(N, m, kinds, n=5):
    """A square whose left, bottom, top and right sides carry boundaries 1..4
    of the list `kinds` (repeated if shorter)."""
    every = {"wall": (E.BC_EULER_WALL, []), "copy": (E.BC_COPY, []),
             "inflow": (E.BC_EULER_INFLOW, [0.4, 20.0, GAMMA, 1.1, 1.2]),
             "dirichlet": (E.BC_EULER_DIRICHLET, [0.9, 0.2, -0.1, 0.0 if m == 4 else 0.1, GAMMA, 0.8])}
    mesh = E.structured_mesh(n, 0.0, 1.0, 0.0, 1.0, 0.1, 3, False)
    tags = np.zeros((n, n, 2, 3), np.int32)
    tags[:, 0, 1, 2], tags[0, :, 0, 0], tags[n - 1, :, 1, 1], tags[:, n - 1, 0, 1] = 1, 2, 3, 4
    mesh = E.MeshData(mesh.VX, mesh.VY, mesh.EToV, mesh.vert_id, tags.reshape(-1, 3))
    bcs = [every[kinds[i % len(kinds)]] for i in range(4)]
    eqn = E.EQN_EULER4 if m == 4 else E.EQN_EULER5
    return Case(mesh, E.Params(N, eqn, gas_gamma=GAMMA, bcs=bcs), "+".join(kinds))


def subsonic_state(case, seed=1):
    """A uniform subsonic flow with 1% noise at the nodes."""
    g = np.random.default_rng(seed)
    q = np.zeros(case.shape)
    q[..., 0], q[..., 1], q[..., 2] = 1.0, 0.3, -0.2
    if case.params.m == 5:
        q[..., 3] = 0.1
    q[..., -1] = 1.0 / (GAMMA - 1) + 0.5 * (0.09 + 0.04)
    return q * (1.0 + 1e-2 * g.standard_normal(q.shape))


def check_dot_product(q, rhs, adjoint, seed=9, zero=None):
    """w . J v from central differences of rhs() against v . J^T w."""
    g = np.random.default_rng(seed)
    v, w = g.standard_normal(q.shape), g.standard_normal(q.shape)
    if zero is not None:
        v[..., zero] = 0.0
    eps = 1e-6
    lhs = np.sum((rhs(q + eps * v) - rhs(q - eps * v)) / (2 * eps) * w)
    r = np.sum(v * adjoint(q, w))
    # central differences: eps^2 of the curvature, and the rounding of the two
    # values, 1e-16 / eps
    assert abs(lhs - r) <= 1e-7 * abs(lhs), (lhs, r)


KINDS = [("wall",), ("inflow",), ("dirichlet",), ("copy",), ("inflow", "wall", "dirichlet", "copy")]
