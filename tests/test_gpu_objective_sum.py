"""The objective's sum over many partials: more than one block of the packing
kernel, with every partial in, some and none, against a sum of the cubature
values element by element."""
import numpy as np
import pytest

from apollo_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [363, 512])     # 4118 and 8192 partials of 64 elements
def test_objective_of_many_partials(n):
    mesh = E.structured_mesh(n, -5.0, 5.0, -5.0, 5.0, 0.1, 7, True)
    eng = E.Engine(mesh, E.Params(1, E.EQN_EULER4, gas_gamma=1.4))
    q = np.random.default_rng(n).uniform(0.5, 1.5, (mesh.K, 3, 4))
    V, w = E.host_operator(1, 0).reshape(-1, 3), E.host_operator(1, 5)
    r, s = (V @ E.host_operator(1, k) for k in (8, 9))
    vx, vy = mesh.VX[mesh.EToV], mesh.VY[mesh.EToV]
    x, y = (0.5 * (-p[:, :1] * (r + s) + p[:, 1:2] * (1 + r) + p[:, 2:] * (1 + s)) for p in (vx, vy))
    J = ((vx[:, 1] - vx[:, 0]) * (vy[:, 2] - vy[:, 0]) - (vx[:, 2] - vx[:, 0]) * (vy[:, 1] - vy[:, 0])) / 4
    for radius in (8.0, 2.0, 0.0):
        inside = (x - 0.2) ** 2 + (y + 0.3) ** 2 < radius ** 2
        ref = float(np.sum(w * J[:, None] * inside * (q[..., 1] @ V.T) ** 2))
        got = eng.objective_disc_sq(q, 1, 0.2, -0.3, radius)
        assert got == eng.objective_disc_sq(q, 1, 0.2, -0.3, radius)
        assert abs(got - ref) <= 1e-12 * ref
    eng.close()
