"""What a user of the engine has it do, as measured calls.

A case is one call through apollo_amd.engine on a structured triangle mesh of
n x n x 2 elements (K = 2 n^2, vertices jittered): Apollo's RHS as its step()
asks for it, LSERK4 steps, one output frame of Apollo's own stepping with the
limiter, the limiter alone, the adjoint RHS, the reverse LSERK4, and the
objective with its gradient.  Sizes, orders, fluxes and precisions are those
of the repository's workloads (apollo_amd/workloads.py), of its benchmark legs
and of Apollo's decks (tests/cases.py), and others of the same ranges.

Plans: the mesh and the engine handle, as a solver keeps them for a whole run.
Inputs: states and adjoint weights drawn from the seed.  Each pass starts from
the same inputs, so a stepper's pass first copies the initial state into its
work tensor, as a program does that starts several runs from one state.
"""
import math

import numpy as np
import torch

from apollo_amd import engine as E

EQNS = {"euler4": E.EQN_EULER4, "euler5": E.EQN_EULER5, "phmaxwell8": E.EQN_PHMAXWELL8,
        "tm3": E.EQN_MAXWELL_TM3}
FLUXES = {"lf": E.FLUX_LF, "hll": E.FLUX_HLL, "upwind": E.FLUX_UPWIND}
PRECISIONS = {"fp64": E.PREC_FP64, "fp32": E.PREC_FP32_MFMA, "bf16x3": E.PREC_BF16X3}
NC = (12, 19, 36, 54, 73, 93, 118, 145)      # cubature points of order 1..8
GAMMA = 1.4
MACH, PRESSURE = 3.0, 5.0                    # the shock decks' inflow (rho = gamma)
LIMITER = (GAMMA, 1e-2, 1e-2)                # the shock decks' limiter block
DISC = (0, 0.2, -0.3, 1.5)                   # objective: variable, centre, radius


def listed():
    return [
        # Apollo's own step(): one RHS with its suggested dt, on host arrays as a PETSc Vec hands
        # them over.  The size of its circular-pulse deck (P_ORDER = 1, HLL, walls).
        {"name": "step_host_euler5_N1", "op": "rhs", "eqn": "euler5", "n": 41, "N": 1, "flux": "hll",
         "bc": "wall", "where": "host", "precision": "fp64"},
        # one output frame of a shock deck (P_ORDER = 1, HLL, limiter, inflow / walls / outflow, about
        # 16 thousand elements in a generator's order): init's dt, then TSSSP under Apollo's dt control
        {"name": "frame_limited_N1", "op": "frame", "eqn": "euler5", "n": 89, "N": 1, "flux": "hll",
         "bc": "channel", "steps": 6, "numbering": "front", "precision": "fp64"},
        # the small Euler vortex of the benchmark: LSERK4 steps of a mesh that does not fill the card
        {"name": "vortex_64_N3_fp64", "op": "lserk4", "eqn": "euler4", "n": 64, "N": 3, "flux": "lf",
         "bc": "periodic", "steps": 10, "precision": "fp64"},
        # the benchmark's headline: Maxwell TM cavity, nodal form
        {"name": "tm_256_N5_fp64", "op": "lserk4", "eqn": "tm3", "n": 256, "N": 5, "flux": "upwind",
         "bc": "tm", "steps": 4, "precision": "fp64"},
        # the high-order Maxwell workload in FP32-MFMA
        {"name": "tm_384_N8_fp32", "op": "lserk4", "eqn": "tm3", "n": 384, "N": 8, "flux": "upwind",
         "bc": "tm", "steps": 2, "precision": "fp32"},
        # the largest workload: Euler vortex, cubature form, FP64
        {"name": "vortex_512_N4_fp64", "op": "lserk4", "eqn": "euler4", "n": 512, "N": 4, "flux": "lf",
         "bc": "periodic", "steps": 2, "precision": "fp64"},
        # the same equations in split-BF16x3 at an odd size, for a run that trades accuracy
        {"name": "vortex_301_N4_bf16x3", "op": "lserk4", "eqn": "euler4", "n": 301, "N": 4, "flux": "lf",
         "bc": "periodic", "steps": 2, "precision": "bf16x3"},
        # Apollo's 8-variable Maxwell system, one RHS with its suggested dt on device tensors
        {"name": "rhs_phmaxwell8_N4", "op": "rhs", "eqn": "phmaxwell8", "n": 150, "N": 4, "flux": "lf",
         "bc": "pec", "where": "device", "precision": "fp64"},
        # the limiter by itself, as a caller of apl_rhs applies it, on the benchmark's mesh
        {"name": "limit_512_N4", "op": "limit", "eqn": "euler5", "n": 512, "N": 4, "flux": "hll",
         "bc": "wall", "precision": "fp64"},
        # one transposed RHS (a sensitivity or an implicit solve's operator) of an odd, middling mesh
        {"name": "adjoint_rhs_euler5_N2", "op": "adjoint_rhs", "eqn": "euler5", "n": 101, "N": 2,
         "flux": "lf", "bc": "periodic", "precision": "fp64"},
        # the reverse LSERK4 of the adjoint workload, checkpointed
        {"name": "reverse_256_N3", "op": "reverse", "eqn": "euler4", "n": 256, "N": 3, "flux": "lf",
         "bc": "periodic", "steps": 8, "ckpt": 4, "precision": "fp64"},
        # that workload's objective and its gradient, which start every reverse sweep
        {"name": "objective_256_N3", "op": "objective", "eqn": "euler4", "n": 256, "N": 3, "flux": "lf",
         "bc": "periodic", "precision": "fp64"},
    ]


def draw(rng):
    op = rng.choice(["rhs", "rhs", "lserk4", "lserk4", "lserk4", "frame", "limit", "adjoint_rhs",
                     "reverse", "objective"])
    c = {"op": op, "precision": "fp64"}
    if op in ("frame", "limit"):
        c["eqn"], c["N"] = rng.choice(["euler5", "euler5", "euler4"]), rng.choice([1, 1, 2, 3, 4])
    elif op in ("reverse", "objective"):
        c["eqn"], c["N"] = rng.choice(["euler4", "euler4", "tm3"]), rng.randint(1, 5)
    elif op == "adjoint_rhs":
        c["eqn"], c["N"] = rng.choice(["euler4", "euler5", "tm3"]), rng.randint(1, 5)
    else:
        c["eqn"], c["N"] = rng.choice(["euler4", "euler5", "tm3", "tm3", "phmaxwell8"]), rng.randint(1, 8)
    if op == "lserk4":
        c["precision"] = rng.choice(["fp64", "fp64", "fp32", "bf16x3"])
    # n over a logarithm, up to where the state has the largest listed one's values
    c["steps"] = {"lserk4": rng.randint(1, 4), "frame": rng.randint(2, 5), "reverse": rng.randint(2, 6)}.get(op, 1)
    m, Np = E.NVARS[EQNS[c["eqn"]]], (c["N"] + 1) * (c["N"] + 2) // 2
    most = 512 * 512 * 60 * (0.5 if op in ("reverse", "adjoint_rhs", "frame") else 1.0)
    most /= c["steps"] * (3.0 if op == "frame" else 1.0) * (1.0 + 0.15 * max(0, c["N"] - 4))
    top = max(24, min(512, int(math.sqrt(most / (Np * m)))))
    c["n"] = int(round(math.exp(rng.uniform(math.log(12), math.log(top)))))
    if op == "reverse":
        c["ckpt"] = rng.randint(1, c["steps"])
    if c["eqn"] in ("tm3", "phmaxwell8"):
        c["flux"] = rng.choice(["lf", "upwind"]) if c["eqn"] == "tm3" else "lf"
        c["bc"] = rng.choice(["tm", "pec"])
    elif op in ("frame", "limit"):
        c["flux"], c["bc"] = rng.choice(["hll", "hll", "lf"]), rng.choice(["channel", "wall"])
    elif op == "rhs":
        c["flux"], c["bc"] = rng.choice(["lf", "hll"]), rng.choice(["periodic", "wall", "channel"])
    else:
        c["flux"], c["bc"] = "lf", "periodic"
    if op == "rhs":
        c["where"] = rng.choice(["device", "device", "host"])
    c["numbering"] = rng.choice(["rows", "front"])
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _euler(c):
    return c["eqn"] in ("euler4", "euler5")


def _extent(c):
    """The domain: Maxwell on the unit square, the vortex on a square around the origin."""
    if not _euler(c):
        return 0.0, 1.0
    half = 5.0 if c["n"] <= 256 else 10.0
    return -half, half


def _mesh(c):
    x0, x1 = _extent(c)
    n, periodic = c["n"], c["bc"] == "periodic"
    m = E.structured_mesh(n, x0, x1, x0, x1, 0.1, 7 + n, periodic)
    etov, tags = m.EToV, m.face_tag
    if c["bc"] == "channel":            # tags 1..4: inflow on the left, bottom, top, outflow
        tags = np.zeros((n, n, 2, 3), np.int32)
        tags[:, 0, 1, 2], tags[0, :, 0, 0] = 1, 2
        tags[n - 1, :, 1, 1], tags[:, n - 1, 0, 1] = 3, 4
        tags = tags.reshape(-1, 3)
    if c.get("numbering") == "front":   # a mesh generator's order: neighbours near, but not in rows
        keys = np.arange(m.K) + np.random.default_rng(n).uniform(0, 96, m.K)
        order = np.argsort(keys)
        etov, tags = etov[order], tags[order]
    return E.MeshData(m.VX, m.VY, etov, m.vert_id, tags)


def _bcs(c):
    wall, copy = (E.BC_EULER_WALL, []), (E.BC_COPY, [])
    inflow = (E.BC_EULER_INFLOW, [MACH, 0.0, GAMMA, PRESSURE, GAMMA])
    return {"periodic": [], "wall": [wall], "channel": [inflow, wall, wall, copy],
            "tm": [(E.BC_MAXWELL_TM, [])], "pec": [(E.BC_PEC, [])]}[c["bc"]]


def _params(c):
    limiter = LIMITER if c["op"] in ("frame", "limit") else None
    ph = {"chi": 1.0, "gamma_ph": 1.0} if c["eqn"] == "phmaxwell8" else {}
    return E.Params(c["N"], EQNS[c["eqn"]], flux=FLUXES[c["flux"]], precision=PRECISIONS[c["precision"]],
                    gas_gamma=GAMMA, bcs=_bcs(c), limiter=limiter, **ph)


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _nodes(c, mesh):
    """Node coordinates x, y [K][Np]: the affine image of the reference nodes."""
    d = _device()
    r, s = (torch.from_numpy(E.host_operator(c["N"], w)).to(d) for w in (8, 9))
    v = torch.from_numpy(mesh.EToV.astype(np.int64)).to(d)
    out = []
    for V in (mesh.VX, mesh.VY):
        p = torch.from_numpy(V).to(d)[v]
        out.append(0.5 * (-p[:, :1] * (r + s) + p[:, 1:2] * (1 + r) + p[:, 2:] * (1 + s)))
    return out


def _modes(g, x, y, L, count=16):
    """A smooth random field of `count` Fourier modes of the square, of order 1."""
    out = torch.zeros_like(x)
    for _ in range(count):
        k = g.integers(1, 6, 2)
        a, p1, p2 = g.standard_normal() / math.sqrt(count), g.uniform(0, 2 * np.pi), g.uniform(0, 2 * np.pi)
        out += a * torch.sin(2 * np.pi * k[0] / L * x + p1) * torch.cos(2 * np.pi * k[1] / L * y + p2)
    return out


def _state(c, x, y, seed):
    g = np.random.default_rng(seed)
    x0, x1 = _extent(c)
    L = x1 - x0
    if not _euler(c):
        comps = [_modes(g, x, y, 2 * L, 6) for _ in range(E.NVARS[EQNS[c["eqn"]]])]
        return torch.stack(comps, -1).contiguous()
    if c["bc"] == "channel":            # the shock decks' uniform Mach flow, with smooth 10% waves on it
        w = [0.1 * torch.tanh(_modes(g, x, y, L, 4)) for _ in range(4)]
        rho, p = GAMMA * (1 + w[0]), PRESSURE * (1 + w[3])
        u, v = MACH * math.sqrt(PRESSURE) * (1 + w[1]), w[2]
    else:                               # the isentropic vortex, its centre and strength from the seed
        beta, cx, cy = g.uniform(4.5, 5.5), g.uniform(-1, 1), g.uniform(-1, 1)
        xs, ys = torch.remainder(x - cx + L / 2, L) - L / 2, torch.remainder(y - cy + L / 2, L) - L / 2
        ex = torch.exp(1 - xs * xs - ys * ys)
        rho = (1 - (GAMMA - 1) * beta ** 2 * ex * ex / (16 * GAMMA * np.pi ** 2)) ** (1 / (GAMMA - 1))
        p = rho ** GAMMA
        u, v = 1 - beta * ex * ys / (2 * np.pi), beta * ex * xs / (2 * np.pi)
        rho = rho * (1 + 1e-3 * _modes(g, x, y, L, 4))
    e = p / (GAMMA - 1) + 0.5 * rho * (u * u + v * v)
    comps = [rho, rho * u, rho * v] + ([torch.zeros_like(rho)] if c["eqn"] == "euler5" else []) + [e]
    return torch.stack(comps, -1).contiguous()


def _cfl(c):
    return 1.0 / (2 * c["N"] + 1)


def _dt(c):
    """A step well inside the stability limit, in closed form."""
    x0, x1 = _extent(c)
    speed = 1.0 if not _euler(c) else 3.5 if c["bc"] != "channel" else 10.0
    return 0.15 * (x1 - x0) / c["n"] / (speed * (c["N"] + 1) ** 2)


def _inputs(c, seed):
    mesh = _mesh(c)
    x, y = _nodes(c, mesh)
    q = _state(c, x, y, seed)
    lam = None
    if c["op"] in ("adjoint_rhs", "reverse"):
        g = torch.Generator(device=q.device).manual_seed(seed)
        lam = torch.randn(q.shape, dtype=torch.float64, device=q.device, generator=g)
    return mesh, q, lam


def prepare(case, seed):
    c = case
    mesh, q, lam = _inputs(c, seed)
    s = {"case": c, "eng": E.Engine(mesh, _params(c)), "q": q, "lam": lam, "dt": _dt(c)}
    if c.get("where") == "host":
        s["q"] = q.cpu().numpy()
        s["out"] = np.zeros_like(s["q"])
    else:
        s["out"] = torch.zeros_like(q)
    if c["op"] == "reverse":
        s["qT"] = torch.zeros_like(q)
    torch.cuda.synchronize()
    return s


def run(state):
    s, c, eng = state, state["case"], state["eng"]
    op, q, out = c["op"], s["q"], s["out"]
    if op == "rhs":
        return out, eng.rhs(0.0, q, out, cfl=_cfl(c))
    if op == "lserk4":
        out.copy_(q)
        eng.lserk4(0.0, s["dt"], c["steps"], out)
        return out
    if op == "frame":
        out.copy_(q)
        dt0 = eng.initial_dt(q, _cfl(c))
        dts = eng.ssp_advance(0.0, (c["steps"] - 0.5) * dt0, dt0, _cfl(c), out, max_steps=1000)
        return out, dt0, dts
    if op == "limit":
        eng.limit(q, out)
        return out
    if op == "adjoint_rhs":
        eng.adjoint_rhs(0.0, q, s["lam"], out)
        return out
    if op == "reverse":
        eng.lserk4_adjoint(0.0, s["dt"], c["steps"], c["ckpt"], q, s["lam"], out, qT=s["qT"])
        return out, s["qT"]
    return eng.objective_disc_sq(q, *DISC, dJdq=out), out


def work(case):
    """Bytes: a state (FP64) each time a stage has to read or write one, since every stage needs its
    neighbours' results, and 136 B of geometry and connectivity per element.  Flops: the contractions
    of the form that the equations allow (nodal for the linear fluxes, cubature for Euler), unpadded."""
    c = case
    K, N, m = 2 * c["n"] ** 2, c["N"], E.NVARS[EQNS[c["eqn"]]]
    Np, Nf, Ng, Nc = (N + 1) * (N + 2) // 2, 3 * (N + 1), 6 * (N + 1), NC[N - 1]
    S, G = K * Np * m * 8, K * 136
    if _euler(c):
        fwd = 2 * m * K * (3 * Nc * Np + 2 * Ng * (N + 1) + Ng * Np)
        adj = 2 * m * K * (4 * Nc * Np + 3 * Ng * (N + 1) + Ng * Np)
    else:
        fwd = adj = 2 * m * K * (2 * Np * Np + Nf * Np)
    op, st = c["op"], c["steps"] if "steps" in c else 1
    if op == "rhs":
        return {"bytes": 2 * S + G, "flops": fwd}
    if op == "lserk4":
        return {"bytes": 5 * st * (4 * S + G), "flops": 5 * st * fwd}
    if op == "frame":      # per stage the limiter and the RHS, each reading and writing the state
        return {"bytes": S + 5 * st * (4 * S + 2 * G), "flops": 5 * st * fwd}
    if op == "limit":
        return {"bytes": 2 * S + G, "flops": 100 * K * m}
    if op == "adjoint_rhs":
        return {"bytes": 3 * S + G, "flops": adj}
    if op == "reverse":    # a forward stage, then a reverse stage that updates two adjoint states
        return {"bytes": 5 * st * (4 * S + G) + 5 * st * (5 * S + G), "flops": 5 * st * (fwd + adj)}
    return {"bytes": 2 * S + G, "flops": 4 * Nc * Np * K}


# ---------------------------------------------------------------------------
# the same values in plain 64-bit torch
# ---------------------------------------------------------------------------
# The element tables (reference nodes, cubature and edge-Gauss operators) define the discretisation
# and are taken as data; everything computed from them is plain torch.

class _Plain:
    def __init__(self, c, mesh, d):
        self.c, self.N, self.m = c, c["N"], E.NVARS[EQNS[c["eqn"]]]
        t = lambda w: torch.from_numpy(E.host_operator(c["N"], w)).to(d)  # noqa: E731
        self.V, self.Dr, self.Ds, self.If, self.VVT, self.w, self.gw, self.r, self.s = (
            t(w) for w in (0, 1, 2, 3, 4, 5, 7, 8, 9))
        self.Ng, self.K, self.Np = self.gw.numel(), mesh.K, self.r.numel()
        self.Wr = self.VVT @ (self.Dr * self.w[:, None]).T
        self.Ws = self.VVT @ (self.Ds * self.w[:, None]).T
        self.Wf = self.VVT @ (self.If * self.gw.repeat(3)[:, None]).T
        v = torch.from_numpy(mesh.EToV.astype(np.int64)).to(d)
        self.vx, self.vy = torch.from_numpy(mesh.VX).to(d)[v], torch.from_numpy(mesh.VY).to(d)[v]
        x, y = self.vx, self.vy
        xr, xs, yr, ys = ((p[:, i] - p[:, 0]) / 2 for p, i in ((x, 1), (x, 2), (y, 1), (y, 2)))
        self.J = xr * ys - xs * yr
        self.jrx, self.jsx, self.jry, self.jsy = ys, -yr, -xs, xr
        ex, ey = x[:, [1, 2, 0]] - x, y[:, [1, 2, 0]] - y
        L = torch.sqrt(ex * ex + ey * ey)
        self.nx, self.ny, self.sj = ey / L, -ex / L, L / 2
        l1, l2, l3 = L[:, 0], L[:, 1], L[:, 2]
        sp = (l1 + l2 + l3) / 2
        self.dtscale = float((torch.sqrt((sp * (sp - l1) * (sp - l2) * (sp - l3)).abs()) / sp).min())
        self.rmin = float((self.r[1] - self.r[0]).abs())
        # faces: neighbour element and face, or -1 and the tag
        ids = mesh.vert_id if mesh.vert_id is not None else np.arange(mesh.Nv)
        e = ids[mesh.EToV][:, [[0, 1], [1, 2], [2, 0]]].reshape(-1, 2).astype(np.int64)
        key = np.minimum(e[:, 0], e[:, 1]) * mesh.Nv + np.maximum(e[:, 0], e[:, 1])
        o = np.argsort(key, kind="stable")
        same = np.nonzero(key[o][1:] == key[o][:-1])[0]
        nbr = np.full(3 * mesh.K, -1, np.int64)
        nbr[o[same]], nbr[o[same + 1]] = o[same + 1], o[same]
        self.nbr = torch.from_numpy(nbr).to(d).reshape(-1, 3)       # 3 element + face
        self.inside = self.nbr >= 0
        tag = mesh.face_tag.astype(np.int64)      # Apollo: an element's last tagged face names them all
        for f in (1, 2):
            tag[:, f] = np.where(tag[:, f] == 0, tag[:, f - 1], tag[:, f])
        self.tag = torch.from_numpy(np.repeat(tag[:, 2:], 3, 1)).to(d)
        rn, sn = self.r.cpu().numpy(), self.s.cpu().numpy()
        on = [(np.nonzero(np.abs(1 + sn) < 1e-9)[0], rn), (np.nonzero(np.abs(rn + sn) < 1e-9)[0], sn),
              (np.nonzero(np.abs(1 + rn) < 1e-9)[0], -sn)]
        self.fmask = [[int(i) for i in ix[np.argsort(k[ix])]] for ix, k in on]

    # -- fluxes ------------------------------------------------------------
    def flux(self, q):
        """F, G and |u| + c (or None) of states [..., m]."""
        if self.c["eqn"] == "tm3":
            a, b, h = q.unbind(-1)
            z = torch.zeros_like(a)
            return torch.stack([-h, z, -a], -1), torch.stack([b, a, z], -1), None
        if self.c["eqn"] == "phmaxwell8":       # c0 = chi = gamma = 1
            ex, ey, ez, bx, by, bz, ph, ps = q.unbind(-1)
            return (torch.stack([ph, bz, -by, ps, -ez, ey, ex, bx], -1),
                    torch.stack([-bz, ph, bx, ez, ps, -ex, ey, by], -1), None)
        five = self.m == 5
        rho, mu, mv, e = q[..., 0], q[..., 1], q[..., 2], q[..., -1]
        u, v = mu / rho, mv / rho
        w = q[..., 3] / rho if five else torch.zeros_like(rho)
        k2 = u * u + v * v + w * w
        p = (GAMMA - 1) * (e - 0.5 * rho * k2)
        F = [mu, mu * u + p, mu * v] + ([mu * w] if five else []) + [(e + p) * u]
        G = [mv, mv * u, mv * v + p] + ([mv * w] if five else []) + [(e + p) * v]
        return torch.stack(F, -1), torch.stack(G, -1), torch.sqrt(k2) + torch.sqrt(GAMMA * p / rho)

    def exterior(self, q, nx, ny, tag):
        """The boundary's state beyond traces q [F, points, m] of faces with these normals and tags."""
        bc, o = self.c["bc"], q.clone()
        if bc in ("tm", "pec"):
            ez, b = (0, 1) if self.m == 3 else (2, 3)
            o[..., ez] = -q[..., ez]
            if bc == "pec":
                bx, by = q[..., b], q[..., b + 1]
                bn, bt = -bx * nx - by * ny, -bx * ny + by * nx
                o[..., b], o[..., b + 1] = bn * nx - bt * ny, bn * ny + bt * nx
                if self.m == 8:
                    en, et = q[..., 0] * nx + q[..., 1] * ny, q[..., 0] * ny - q[..., 1] * nx
                    o[..., 0], o[..., 1], o[..., 6] = en * nx - et * ny, en * ny + et * nx, -q[..., 6]
            return o
        qn = nx * q[..., 1] + ny * q[..., 2]
        o[..., 1], o[..., 2] = q[..., 1] - 2 * qn * nx, q[..., 2] - 2 * qn * ny
        if self.m == 5:
            o[..., 3] = 0
        if bc == "channel":
            u = MACH * math.sqrt(PRESSURE)
            full = torch.zeros(self.m, dtype=q.dtype, device=q.device)
            full[0], full[1], full[-1] = GAMMA, GAMMA * u, PRESSURE / (GAMMA - 1) + 0.5 * GAMMA * u * u
            o = torch.where((tag == 1)[:, None, None], full.expand_as(q), o)
            o = torch.where((tag == 4)[:, None, None], q, o)
        return o

    def star(self, qM, qP, nx, ny):
        """The numerical flux and the fastest speed at points with normals nx, ny [..., 1]."""
        if self.c["flux"] == "hll":
            return self.hll(qM, qP, nx, ny)
        FM, GM, cM = self.flux(qM)
        FP, GP, cP = self.flux(qP)
        lam = torch.ones_like(qM[..., 0]) if cM is None else torch.maximum(cM, cP)
        nX, nY = nx[..., None], ny[..., None]
        f = 0.5 * (nX * (FM + FP) + nY * (GM + GP) + lam[..., None] * (qM - qP))
        if self.c["flux"] == "upwind":
            jb = nx * (qM[..., 1] - qP[..., 1]) + ny * (qM[..., 2] - qP[..., 2])
            f = torch.stack([f[..., 0], f[..., 1] - 0.5 * nx * jb, f[..., 2] - 0.5 * ny * jb], -1)
        return f, lam

    def hll(self, qM, qP, nx, ny):
        def rot(q):
            o = q.clone()
            o[..., 1], o[..., 2] = nx * q[..., 1] + ny * q[..., 2], -ny * q[..., 1] + nx * q[..., 2]
            return o

        a, b = rot(qM), rot(qP)
        FM, _, cM = self.flux(a)
        FP, _, cP = self.flux(b)

        def prim(q):
            rho, e = q[..., 0], q[..., -1]
            w = q[..., 3] / rho if self.m == 5 else torch.zeros_like(rho)
            u, v = q[..., 1] / rho, q[..., 2] / rho
            p = (GAMMA - 1) * (e - 0.5 * rho * (u * u + v * v + w * w))
            return torch.sqrt(rho), u, v, w, (e + p) / rho, torch.sqrt(GAMMA * p / rho)

        rM, uM, vM, wM, HM, aM = prim(a)
        rP, uP, vP, wP, HP, aP = prim(b)
        u, v, w, H = ((rM * s + rP * t) / (rM + rP) for s, t in ((uM, uP), (vM, vP), (wM, wP), (HM, HP)))
        cc = torch.sqrt((GAMMA - 1) * (H - 0.5 * (u * u + v * v + w * w)))
        SL, SR = torch.minimum(uM - aM, u - cc), torch.maximum(uP + aP, u + cc)
        t1 = (SR.clamp(max=0) - SL.clamp(max=0)) / (SR - SL)
        t3 = (SR * SL.abs() - SL * SR.abs()) / (2 * (SR - SL))
        f = t1[..., None] * FP + (1 - t1)[..., None] * FM - t3[..., None] * (b - a)
        o = f.clone()
        o[..., 1], o[..., 2] = nx * f[..., 1] - ny * f[..., 2], ny * f[..., 1] + nx * f[..., 2]
        if self.m == 5:
            o[..., 3] = 0
        return o, torch.maximum(cM, cP)

    # -- the RHS -----------------------------------------------------------
    def rhs(self, q):
        """The RHS of state q [K][Np][m] and the fastest face speed."""
        K, Ng, m = self.K, self.Ng, self.m
        tr = torch.matmul(self.If, q).reshape(3 * K, Ng, m)
        back = tr.flip(1)
        nx, ny = self.nx.reshape(-1, 1).expand(-1, Ng), self.ny.reshape(-1, 1).expand(-1, Ng)
        nb, inside = self.nbr.reshape(-1), self.inside.reshape(-1)
        qP = back[nb.clamp(min=0)]
        if not bool(inside.all()):
            at = torch.nonzero(~inside)[:, 0]
            qP = qP.index_copy(0, at, self.exterior(tr[at], nx[at], ny[at], self.tag.reshape(-1)[at]))
        f, lam = self.star(tr, qP, nx, ny)
        f = (f * self.sj.reshape(-1, 1, 1)).reshape(K, 3 * Ng, m)
        out = []
        for k in range(0, K, 65536):
            e = slice(k, k + 65536)
            F, G, _ = self.flux(torch.matmul(self.V, q[e]))
            g = lambda z: z[e, None, None]  # noqa: E731
            v = torch.matmul(self.Wr, g(self.jrx) * F + g(self.jry) * G)
            v = v + torch.matmul(self.Ws, g(self.jsx) * F + g(self.jsy) * G)
            out.append((v - torch.matmul(self.Wf, f[e])) / g(self.J))
        return torch.cat(out), lam.max()

    def suggested(self, speed):
        return 2.0 / 3.0 * _cfl(self.c) * self.dtscale * (self.rmin / float(speed))

    A = (0.0, -567301805773.0 / 1357537059087.0, -2404267990393.0 / 2016746695238.0,
         -3550918686646.0 / 2091501179385.0, -1275806237668.0 / 842570457699.0)
    B = (1432997174477.0 / 9575080441755.0, 5161836677717.0 / 13612068292357.0,
         1720146321549.0 / 2090206949498.0, 3134564353537.0 / 4481467310338.0,
         2277821191437.0 / 14882151754819.0)

    def stages(self, q, dt, steps):
        """LSERK4: every stage's input, then the last state."""
        res, out = torch.zeros_like(q), []
        for _ in range(steps):
            for a, b in zip(self.A, self.B):
                out.append(q)
                res = a * res + dt * self.rhs(q)[0]
                q = q + b * res
        return out, q

    def transposed(self, q, lam):
        with torch.enable_grad():
            x = q.detach().requires_grad_(True)
            return torch.autograd.grad(self.rhs(x)[0], x, lam)[0]

    # -- Apollo's limiter ------------------------------------------------------
    @staticmethod
    def prim(q):
        rho = q[..., 0]
        ke = 0.5 * (q[..., 1] ** 2 + q[..., 2] ** 2 + q[..., 3] ** 2) / rho
        return torch.stack([rho, q[..., 1] / rho, q[..., 2] / rho, q[..., 3] / rho,
                            (GAMMA - 1) * (q[..., 4] - ke)], -1)

    def beyond(self, q5, f):
        """The boundary state of face f seen from 5-variable states [K][5]."""
        keep, self.m = self.m, 5
        o = self.exterior(q5[:, None], self.nx[:, f, None], self.ny[:, f, None], self.tag[:, f])[:, 0]
        self.m = keep
        return o

    def limit(self, q):
        q5 = q if self.m == 5 else torch.cat([q[..., :3], torch.zeros_like(q[..., :1]), q[..., 3:]], -1)
        ave = 0.5 * torch.linalg.inv(self.VVT).sum(0)
        avg = torch.einsum("n,knc->kc", ave, q5)
        xc, yc = (self.vx * ave[:3]).sum(1), (self.vy * ave[:3]).sum(1)
        A = 2.0 / 3.0 * self.J * ave[:3].sum()
        el = torch.div(self.nbr, 3, rounding_mode="floor")
        fa = self.nbr - 3 * el
        src, cur = [], torch.arange(self.K, device=q.device)
        for f in range(3):
            cur = torch.where(self.inside[:, f], el[:, f], cur)
            src.append(cur)
        P0, P, X, Y, AA = self.prim(avg), [], [], [], []
        for f in range(3):
            i, ie = self.inside[:, f], el[:, f].clamp(min=0)
            h1 = 2 * A / self.sj[:, f]
            X.append(torch.where(i, xc[ie], xc + 2 * self.nx[:, f] * h1))
            Y.append(torch.where(i, yc[ie], yc + 2 * self.ny[:, f] * h1))
            AA.append(A + torch.where(i, A[ie], torch.zeros_like(A)))
            P.append(self.prim(torch.where(i[:, None], avg[ie], self.beyond(avg, f))))
        F, nfp, ends = self.fmask, self.N + 1, []
        for fi, ni in ((0, 0), (0, nfp - 1), (1, nfp - 1)):
            f, j = divmod(F[fi][ni], nfp)
            far = torch.tensor([F[g][nfp - 1 - j] for g in range(3)], device=q.device)
            i, ie = self.inside[:, f], el[:, f].clamp(min=0)
            mine, other = q5[:, F[f][j]], q5[ie, far[fa[:, f].clamp(min=0)]]
            out = torch.where(i[:, None], other, self.beyond(q5[src[f], F[f][j]], f))
            ends.append(self.prim(0.5 * (out + mine)))
        a, b, e = ends
        x, y = self.vx, self.vy
        d12, d23 = (x[:, 1] - x[:, 0], y[:, 1] - y[:, 0]), (x[:, 2] - x[:, 1], y[:, 2] - y[:, 1])
        gx, gy = [], []
        for f, (d, jump) in enumerate(((d12, a - b), (d23, b - e), (d23, e - a))):
            dp, c1 = P[f] - P0, lambda z: z[:, None]  # noqa: E731
            gx.append(0.5 * (dp * c1(d[1]) + jump * c1(Y[f] - yc)) / c1(AA[f]))
            gy.append(-0.5 * (dp * c1(d[0]) + jump * c1(X[f] - xc)) / c1(AA[f]))
        tot = sum(AA)[:, None]
        cx, cy = (sum(AA[f][:, None] * g[f] for f in range(3)) / tot for g in (gx, gy))
        hx, hy, g2 = [], [], []
        for f in range(3):
            i, ie = self.inside[:, f, None], el[:, f].clamp(min=0)
            hx.append(torch.where(i, cx[ie], gx[f]))
            hy.append(torch.where(i, cy[ie], gy[f]))
            g2.append(hx[f] ** 2 + hy[f] ** 2)
        fac, eps = g2[0] ** 2 + g2[1] ** 2 + g2[2] ** 2, 1e-14
        w = [(g2[(f + 1) % 3] * g2[(f + 2) % 3] + eps) / (fac + 3 * eps) for f in range(3)]
        Lx, Ly = (sum(w[f] * h[f] for f in range(3)) for h in (hx, hy))
        cr, cs = self.r - (ave * self.r).sum(), self.s - (ave * self.s).sum()
        off = lambda p: 0.5 * ((p[:, 1:2] - p[:, :1]) * cr + (p[:, 2:] - p[:, :1]) * cs)  # noqa: E731
        d = off(x)[..., None] * Lx[:, None] + off(y)[..., None] * Ly[:, None]
        drho, du, dv, dw, dp = d.unbind(-1)
        rho0, u, v, z, p0 = (P0[:, None, c] for c in range(5))
        C = [avg[:, None, c] for c in range(5)]
        low, done = LIMITER[1:], torch.zeros_like(drho, dtype=torch.bool)
        rho = rho0 + drho
        bad = rho < low[0]
        for it in range(4):
            todo = bad & ~done
            drho = torch.where(todo, 0.5 * drho, drho)
            rho = torch.where(todo, rho0 + drho, rho)
            done = done | (todo & (rho > low[0]))
        rho = torch.where(bad & ~done, C[0].expand_as(rho), rho)
        ru, rv, rw = C[1] + rho0 * du + drho * u, C[2] + rho0 * dv + drho * v, C[3] + rho0 * dw + drho * z
        ke = 0.5 * (ru * ru + rv * rv + rw * rw)

        def energy(dp):
            return C[4] + dp / (GAMMA - 1) + 0.5 * drho * (u * u + v * v + z * z) + rho0 * (u * du + v * dv + z * dw)

        en = energy(dp)
        p = (GAMMA - 1) * (en - ke / rho)
        bad, done = p < low[1], torch.zeros_like(done)
        for it in range(4):
            todo = bad & ~done
            dp = torch.where(todo, 0.5 * dp, dp)
            en = torch.where(todo, energy(dp), en)
            done = done | (todo & ((GAMMA - 1) * (en - ke / rho) > low[1]))
        en = torch.where(bad & ~done, p0 / (GAMMA - 1) + ke / rho, en)
        return torch.stack([rho, ru, rv] + ([rw] if self.m == 5 else []) + [en], -1)

    def frame(self, q, steps):
        """init's dt from the Roe speeds, then TSSSP rks2 with five stages under Apollo's dt control."""
        p = self.prim(q if self.m == 5 else torch.cat([q[..., :3], torch.zeros_like(q[..., :1]), q[..., 3:]], -1))
        a = torch.sqrt(GAMMA * p[..., 4] / p[..., 0])
        s = torch.stack([x + k * a for x in (p[..., 1], p[..., 2]) for k in (-1, 0, 1)]).abs().max()
        dt0 = self.suggested(s)
        t, end, nxt, dts = 0.0, (steps - 0.5) * dt0, dt0, []
        while t < end:
            dt = min(nxt, abs(end - t))
            w = q
            for _ in range(4):
                w = self.limit(w)
                w = w + dt / 4 * self.rhs(w)[0]
            w = self.limit(w)
            r, speed = self.rhs(w)
            q = 0.8 * w + dt / 5 * r + 0.2 * q
            nxt, t = min(self.suggested(speed), dt), t + dt
            dts.append(dt)
        return q, dt0, np.array(dts)

    def objective(self, q):
        var, xo, yo, rad = DISC
        r, s = self.V @ self.r, self.V @ self.s                        # the cubature points
        x, y = (0.5 * (-p[:, :1] * (r + s) + p[:, 1:2] * (1 + r) + p[:, 2:] * (1 + s)) for p in (self.vx, self.vy))
        wt = self.w * self.J[:, None] * ((x - xo) ** 2 + (y - yo) ** 2 < rad * rad)
        qc = q[..., var] @ self.V.T
        g = torch.zeros_like(q)
        g[..., var] = (2 * wt * qc) @ self.V
        return float((wt * qc * qc).sum()), g


def exact(case, seed):
    c = case
    with torch.no_grad():
        mesh, q, lam = _inputs(c, seed)
        d = _Plain(c, mesh, q.device)
        op, dt = c["op"], _dt(c)
        if op == "rhs":
            r, speed = d.rhs(q)
            return r, d.suggested(speed)
        if op == "lserk4":
            return d.stages(q, dt, c["steps"])[1]
        if op == "frame":
            return d.frame(q, c["steps"])
        if op == "limit":
            return d.limit(q)
        if op == "adjoint_rhs":
            return d.transposed(q, lam)
        if op == "objective":
            return d.objective(q)
        inputs, qT = d.stages(q, dt, c["steps"])
        qb, rb = lam.clone(), torch.zeros_like(lam)
        for i in reversed(range(len(inputs))):
            rb = rb + d.B[i % 5] * qb
            qb = qb + dt * d.transposed(inputs[i], rb)
            rb = d.A[i % 5] * rb
        return qb, qT
