"""The workloads that the performance of this framework is measured on.

Each case is one piece of work as a user's program has it done through the
package's public entry points: a convection-diffusion solve, time steps, a
batch, a served burst of requests, a matrix product.  prepare() builds what
such a program holds beforehand (hierarchy, coefficients, device vectors),
run() is one pass, and exact() computes the same result with dense 64-bit
element matrices and an unpreconditioned-by-multigrid Krylov solver in torch:
from the package it takes the unknowns' numbering (cell vertices and DOF map)
and nothing else.
"""
import math

import numpy as np
import torch

import parmoon_cmg_amd as pm

# the solver settings of the benchmark configurations (damped Jacobi 3 + 3,
# omega 0.5, exact coarse solve), of the first configuration (2 + 2, omega
# 0.8), and of the reference's shipped input file (SSOR 3 + 3, omega 1)
BENCH = dict(omega=0.5, pre=3, post=3, restart=20, maxit=1000, rel_tol=1e-10)
FIRST = dict(omega=0.8, pre=2, post=2, restart=20, maxit=200, rel_tol=1e-10)
SSOR = dict(smoother=3, omega=1.0, pre=3, post=3, restart=20, maxit=200, rel_tol=1e-10)
SOLVERS = dict(bench=BENCH, first=FIRST, ssor=SSOR)
TAU = 1e-3

# meshes of a batch (m macro bricks per side, refined twice) and of a served
# burst (order, m, levels): uneven, with repeats
BATCH_M = (2, 3, 4, 5, 6, 7, 8, 10, 3, 5, 2, 7)
SERVE = ((1, 2, 3), (2, 2, 3), (1, 3, 4), (1, 5, 3), (2, 3, 3), (1, 7, 3), (1, 2, 4), (2, 5, 2), (1, 3, 3),
         (2, 2, 4), (1, 5, 4), (2, 7, 2), (1, 6, 4), (2, 3, 4), (1, 7, 4), (2, 2, 3))


def listed():
    return [
        # the smallest solve: Poisson with a manufactured source, Q1 16^3, 3 levels, the whole
        # program in launches and latency; the solution goes to the host
        dict(name="cd_q1_16_fp64", kind="cd", order=1, m=1, k0=2, levels=3, fp64=True, solver="first", eps=1.0, conv=0.0,
             supg=False, source="sine", host=True),
        # the reference's own input settings: SSOR in its row order
        dict(name="cd_q1_16_ssor", kind="cd", order=1, m=1, k0=2, levels=3, fp64=True, solver="ssor", eps=0.01, conv=0.7,
             supg=True, source="one", host=True),
        # the headline problem, plain FP64 and mixed precision, solution kept on the device
        dict(name="cd_q2_64_fp64", kind="cd", order=2, m=1, k0=2, levels=5, fp64=True, solver="bench", eps=1e-3, conv=1.145,
             supg=True, source="one", host=False),
        dict(name="cd_q2_64_mixed", kind="cd", order=2, m=1, k0=2, levels=5, fp64=False, solver="bench", eps=1e-3,
             conv=1.145, supg=True, source="one", host=False),
        # the largest mesh of the serving workload, on 3^3 macro bricks
        dict(name="cd_q2_96_mixed", kind="cd", order=2, m=3, k0=1, levels=5, fp64=False, solver="bench", eps=1e-3,
             conv=1.145, supg=True, source="one", host=False),
        # time steps of the transported pulse with re-assembly in every step, both precisions
        dict(name="tcd_q1_128_fp64", kind="tcd", order=1, m=1, k0=3, levels=5, fp64=True, supg=False, steps=3),
        dict(name="tcd_q1_128_mixed", kind="tcd", order=1, m=1, k0=3, levels=5, fp64=False, supg=False, steps=3),
        # the stabilised time steps: element matrices vary from cell to cell
        dict(name="tcd_q2_24_supg_mixed", kind="tcd", order=2, m=3, k0=0, levels=4, fp64=False, supg=True, steps=3),
        # twelve small problems of uneven size solved together
        dict(name="batch_q1_fp64", kind="batch", order=1, levels=3, fp64=True, first=0, count=12),
        # a burst of requests at the serving loop, one request per slot
        dict(name="serve_mixed", kind="serve", fp64=False, first=0, count=16),
        # general hexahedra (deformed 3^3 macro mesh): assembled cell by cell
        dict(name="hex_q2_48_mixed", kind="hex", order=2, m=3, k0=0, levels=5, fp64=False, eps=1e-3, conv=1.145),
        # y = A x on the headline problem's finest matrix, device vectors
        dict(name="matvec_q2_64", kind="matvec", order=2, m=1, k0=2, levels=5, eps=1e-3, conv=1.145),
    ]


def _mesh(rng, lo, hi, order):
    """A mesh m 2^k with lo <= m 2^k <= hi cells per side, log-uniform, at least 2 levels, coarsest at most 8 cells."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    found = []
    for m in (1, 2, 3, 5, 6, 7):
        for k in range(1, 8):
            if lo <= m << k <= hi and not (m == 1 and k < 2):
                found.append((abs((m << k) - n), m, k))
    _, m, k = min(found)
    k0 = 1 if m == 1 else 0
    return dict(order=order, m=m, k0=k0, levels=min(5, k - k0 + 1) if m > 1 else k - k0 + 1)


def draw(rng):
    kind = rng.choice(("cd", "cd", "cd", "tcd", "tcd", "hex", "batch", "serve", "matvec"))
    order = rng.choice((1, 2))
    fp64 = rng.random() < 0.5
    top = 128 // order
    eps = 10 ** rng.uniform(-3, 0)
    if kind == "cd":
        return dict(kind=kind, fp64=fp64, solver="bench", eps=eps, conv=rng.uniform(0.1, 1.2), supg=True, source="one",
                    host=rng.random() < 0.5, **_mesh(rng, 8, top, order))
    if kind == "tcd":
        supg = rng.random() < 0.4
        return dict(kind=kind, fp64=fp64, supg=supg, steps=rng.choice((1, 2, 3)), **_mesh(rng, 8, 24 if supg else top, order))
    if kind == "hex":
        m = _mesh(rng, 8, 48, order)
        return dict(kind=kind, fp64=fp64, eps=eps, conv=rng.uniform(0.1, 1.2), **(m if m["m"] > 1 else dict(m, m=2, k0=0)))
    if kind == "matvec":
        return dict(kind=kind, eps=eps, conv=rng.uniform(0.1, 1.2), **_mesh(rng, 12, top, order))
    if kind == "batch":
        return dict(kind=kind, order=1, levels=3, fp64=fp64, first=rng.randrange(len(BATCH_M)), count=rng.randint(4, 12))
    return dict(kind=kind, fp64=fp64, first=rng.randrange(len(SERVE)), count=rng.randint(6, 16))


# ------------------------------------------------------------------ what a program holds

def _rng(seed):
    return np.random.default_rng(int(seed))


def _coeffs(case, rng):
    """Constant coefficients near the case's: a direction near (1, 0.5, 0.25), f near 1."""
    d = np.array([1.0, 0.5, 0.25]) + 0.2 * rng.uniform(-1, 1, 3)
    b = d / np.linalg.norm(d) * case["conv"]
    return dict(eps=case["eps"] * rng.uniform(0.9, 1.1), b=tuple(float(x) for x in b), supg=int(case.get("supg", True)),
                f_kind=1 if case.get("source") == "sine" else 0, f_val=float(rng.uniform(0.5, 2.0)))


def _tcd_coeffs(case, rng):
    """The rotating field with a Gaussian pulse; SUPG runs carry a source."""
    pulse = np.array([0.3, 0.5, 0.5]) + 0.05 * rng.uniform(-1, 1, 3)
    return dict(eps=1e-4 * rng.uniform(0.9, 1.1), conv_kind=1, rot_c=(0.5, 0.5), pulse_c=tuple(float(x) for x in pulse),
                f_val=1.0 if case["supg"] else 0.0, supg=int(case["supg"]))


def _many_coeffs(count, rng):
    """The uneven problems' coefficients: eps log-uniform, a random direction."""
    out = []
    for _ in range(count):
        d = rng.standard_normal(3)
        b = d / np.linalg.norm(d) * rng.uniform(0.1, 1)
        out.append(dict(eps=float(10 ** rng.uniform(-3, 0)), b=tuple(float(x) for x in b), f_val=1.0, supg=1))
    return out


def _batch_m(case):
    return [BATCH_M[(case["first"] + i) % len(BATCH_M)] for i in range(case["count"])]


def _serve_meshes(case):
    return [SERVE[(case["first"] + i) % len(SERVE)] for i in range(case["count"])]


def _vertices(m, rng):
    """Macro vertices of the unit cube, the interior ones moved."""
    g = np.arange(m + 1, dtype=np.float64)
    k, j, i = np.meshgrid(g, g, g, indexing="ij")
    inner = (i > 0) & (i < m) & (j > 0) & (j < m) & (k > 0) & (k < m)
    d = 0.15 * rng.uniform(-1, 1, i.shape + (3,)) * inner[..., None]
    return ((np.stack([i, j, k], -1) + d) / m).reshape(-1, 3)


def _precision(case):
    return pm.FP64 if case["fp64"] else pm.MIXED


def _problem(case, **kw):
    return pm.Problem(case["order"], case["m"], case["k0"], case["levels"], **kw)


def _fine(P):
    return P.info(P.levels - 1)["ndof"]


class _Solution:
    """The finest level's solution vector of a handle, for torch.as_tensor; it lives as long as the handle."""

    def __init__(self, P):
        self.owner = P
        self.__cuda_array_interface__ = dict(shape=(_fine(P),), typestr="<f8", data=(P.device_ptr(P.levels - 1, 0), False),
                                             version=2)


def _pulse(P, co):
    return P.interp_pulse(P.levels - 1, pm.coeffs(**co))


def prepare(case, seed):
    rng = _rng(seed)
    kind = case["kind"]
    if kind in ("cd", "hex"):
        P = _problem(case, vertices=_vertices(case["m"], rng)) if kind == "hex" else _problem(case)
        co = pm.coeffs(**_coeffs(case, rng))
        sp = pm.solver_params(**SOLVERS[case.get("solver", "bench")], precision=_precision(case))
        x = out = None
        if not case.get("host"):
            x = torch.as_tensor(_Solution(P), device="cuda")
            out = torch.empty_like(x)  # the handle's vector goes with the handle: results are copied out of it
        return dict(kind="solve", P=P, co=co, sp=sp, x=x, out=out)
    if kind == "tcd":
        P = _problem(case)
        co = _tcd_coeffs(case, rng)
        return dict(kind=kind, P=P, co=pm.coeffs(**co), u0=_pulse(P, co), steps=case["steps"],
                    sp=pm.solver_params(**BENCH, precision=_precision(case)))
    if kind == "batch":
        Ps = [pm.Problem(1, m, 0, case["levels"]) for m in _batch_m(case)]
        return dict(kind=kind, Ps=Ps, cos=[pm.coeffs(**c) for c in _many_coeffs(len(Ps), rng)],
                    sp=pm.solver_params(**BENCH, precision=_precision(case)))
    if kind == "serve":
        meshes = _serve_meshes(case)
        srv = pm.Server(max_inflight=len(meshes), max_batch=1)
        s = dict(kind=kind, srv=srv, cos=[pm.coeffs(**c) for c in _many_coeffs(len(meshes), rng)],
                 meshes=[pm.mesh_desc(o, m, 0, lv) for o, m, lv in meshes],
                 n=[(o * (m << (lv - 1)) + 1) ** 3 for o, m, lv in meshes],
                 sp=pm.solver_params(**BENCH, precision=_precision(case)))
        run(s)  # a serving program's hierarchies are resident
        return s
    P = _problem(case)
    P.assemble(pm.coeffs(**_coeffs(case, rng)))
    x = torch.from_numpy(rng.standard_normal(_fine(P))).cuda()
    y = torch.empty_like(x)
    P.synchronize()
    torch.cuda.synchronize()  # the product runs on the handle's stream
    return dict(kind="matvec", P=P, l=P.levels - 1, x=x, y=y)


def run(state):
    s = state
    if s["kind"] == "solve":
        s["P"].assemble(s["co"])
        if s["x"] is None:
            return s["P"].solve(s["sp"])[0]
        s["P"].solve_device(s["sp"])  # waits for the handle's stream
        return s["out"].copy_(s["x"])
    if s["kind"] == "tcd":
        s["P"].tcd_init(s["co"], 0.0, s["u0"])
        for _ in range(s["steps"]):
            s["P"].tcd_step(s["co"], s["sp"], TAU, want_state=False)
        return s["P"].tcd_state()
    if s["kind"] == "batch":
        for P, co in zip(s["Ps"], s["cos"]):
            P.assemble(co)
        pm.solve_batch(s["Ps"], s["sp"])
        return [P.solution() for P in s["Ps"]]
    if s["kind"] == "serve":
        ids = [s["srv"].submit(mesh, co, s["sp"], want_solution=True) for mesh, co in zip(s["meshes"], s["cos"])]
        return [s["srv"].wait(i, n_dof=n)[1] for i, n in zip(ids, s["n"])]
    s["P"].matvec_dev(s["l"], s["x"].data_ptr(), s["y"].data_ptr())
    return s["y"]


# ------------------------------------------------------------------ what a pass cannot do without

def _solve_work(order, n, fp64, its):
    """`its` iterations of FGMRES with a 3 + 3 V-cycle over all levels: per sweep or defect the level's vectors once
    (iterate and rhs read, result written), 2 flops per stencil entry, the Krylov basis read twice per iteration."""
    N = (order * n + 1) ** 3
    s = 8 if fp64 else 4
    sten = 27 if order == 1 else 64
    sweeps = 8 * 8 / 7
    return dict(bytes=its * (sweeps * 3 * s * N + 24 * 8 * N), flops=its * ((sweeps + 1) * 2 * sten + 44) * N)


def work(case):
    kind = case["kind"]
    if kind in ("batch", "serve"):
        sizes = [(1, m << 2) for m in _batch_m(case)] if kind == "batch" else \
            [(o, m << (lv - 1)) for o, m, lv in _serve_meshes(case)]
        each = [_solve_work(o, n, case["fp64"], 20) for o, n in sizes]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    order, n = case["order"], case["m"] << (case["k0"] + case["levels"] - 1)
    if kind == "matvec":
        N = (order * n + 1) ** 3
        return dict(bytes=16 * N, flops=2 * (27 if order == 1 else 64) * N)
    if kind == "tcd":
        w = _solve_work(order, n, case["fp64"], 5)
        return {k: case["steps"] * v for k, v in w.items()}
    return _solve_work(order, n, case["fp64"], 20)


# ------------------------------------------------------------------ the same results in 64 bits

_G = {1: ((-0.6 ** 0.5, 0.0, 0.6 ** 0.5), (5 / 9, 8 / 9, 5 / 9))}
_a, _b = math.sqrt(3 / 7 - 2 / 7 * math.sqrt(1.2)), math.sqrt(3 / 7 + 2 / 7 * math.sqrt(1.2))
_wa, _wb = (18 + math.sqrt(30)) / 36, (18 - math.sqrt(30)) / 36
_G[2] = ((_a, _b, -_b, -_a), (_wa, _wb, _wb, _wa))
_HEX = ((-1, -1, -1), (1, -1, -1), (1, 1, -1), (-1, 1, -1), (-1, -1, 1), (1, -1, 1), (1, 1, 1), (-1, 1, 1))


def _lagrange(p, x):
    if p == 1:
        return [0.5 - 0.5 * x, 0.5 + 0.5 * x], [-0.5, 0.5]
    return [0.5 * x * (x - 1), 1 - x * x, 0.5 * x * (x + 1)], [x - 0.5, -2 * x, x + 0.5]


class _Fem:
    """Element matrices of one mesh level, applied cell by cell."""

    def __init__(self, order, cells, gn, nact, device):
        self.p, self.nact, self.dev = order, nact, device
        self.V = torch.from_numpy(np.ascontiguousarray(cells)).to(device)   # (ncell, 8, 3)
        self.gn = torch.from_numpy(np.ascontiguousarray(gn)).to(device).long()
        self.n = int(gn.max()) + 1
        g, w = _G[order]
        self.pts = [((g[k], g[j], g[i]), w[i] * w[j] * w[k]) for i in range(len(g)) for j in range(len(g))
                    for k in range(len(g))]
        self.chunk = 16384 if order == 2 else 131072

    def _basis(self, r):
        v, d = zip(*(_lagrange(self.p, x) for x in r))
        q = range(self.p + 1)
        phi = [v[0][i] * v[1][j] * v[2][k] for k in q for j in q for i in q]
        dphi = [(d[0][i] * v[1][j] * v[2][k], v[0][i] * d[1][j] * v[2][k], v[0][i] * v[1][j] * d[2][k])
                for k in q for j in q for i in q]
        t = dict(dtype=torch.float64, device=self.dev)
        return torch.tensor(phi, **t), torch.tensor(dphi, **t)

    def _map(self, V, r):
        N = [0.125 * (1 + h[0] * r[0]) * (1 + h[1] * r[1]) * (1 + h[2] * r[2]) for h in _HEX]
        dN = [(0.125 * h[0] * (1 + h[1] * r[1]) * (1 + h[2] * r[2]), 0.125 * h[1] * (1 + h[0] * r[0]) * (1 + h[2] * r[2]),
               0.125 * h[2] * (1 + h[0] * r[0]) * (1 + h[1] * r[1])) for h in _HEX]
        t = dict(dtype=torch.float64, device=self.dev)
        X = torch.einsum("v,cvd->cd", torch.tensor(N, **t), V)
        J = torch.einsum("va,cvd->cda", torch.tensor(dN, **t), V)  # dX_d / dr_a
        c0, c1, c2 = J[:, :, 0], J[:, :, 1], J[:, :, 2]
        rows = [torch.linalg.cross(c1, c2), torch.linalg.cross(c2, c0), torch.linalg.cross(c0, c1)]
        det = (c0 * rows[0]).sum(1)
        return X, torch.stack(rows, 1) / det[:, None, None], det.abs()  # inverse: dr_a / dX_d

    def _conv(self, co, X):
        if co.get("conv_kind"):
            bz = torch.full_like(X[:, 0], 0.1 * math.sin(2 * math.pi * co["t"]))
            return torch.stack([-(X[:, 1] - co["rot_c"][1]), X[:, 0] - co["rot_c"][0], bz], 1)
        return torch.tensor(co.get("b", (0, 0, 0)), dtype=torch.float64, device=self.dev).expand(X.shape)

    def _source(self, co, X, b):
        if not co.get("f_kind"):
            return torch.full_like(X[:, 0], co["f_val"])
        s, c = torch.sin(math.pi * X), torch.cos(math.pi * X)
        u = s[:, 0] * s[:, 1] * s[:, 2]
        grad = math.pi * torch.stack([c[:, 0] * s[:, 1] * s[:, 2], s[:, 0] * c[:, 1] * s[:, 2], s[:, 0] * s[:, 1] * c[:, 2]], 1)
        return co["eps"] * 3 * math.pi ** 2 * u + (b * grad).sum(1)

    def _delta(self, V, co):
        """Per cell: the mesh size in the direction of the convection at the first point."""
        X, _, _ = self._map(V, self.pts[0][0])
        b = self._conv(co, X)
        Vc = V - V.mean(1, keepdim=True)
        size = Vc.abs().amax((1, 2))
        x, y, z = (Vc[:, :, d] / size[:, None] for d in range(3))
        A = torch.stack([torch.ones_like(x), x, y, z, x * y, x * z, y * z, x * y * z], 2)
        eye = torch.eye(8, dtype=torch.float64, device=self.dev).expand_as(A)
        grad = torch.linalg.solve(A, eye)[:, 1:4, :] / size[:, None, None]
        den = torch.einsum("cd,cdv->cv", b, grad).abs().sum(1)
        return 2 * b.norm(dim=1) / den

    def matrices(self, co, what):
        """(element matrices, rhs): "A" convection-diffusion, "M" mass, "K" the SUPG time-derivative matrix."""
        nb = self.gn.shape[1]
        E = torch.empty((len(self.V), nb, nb), dtype=torch.float64, device=self.dev)
        rhs = torch.zeros(self.n, dtype=torch.float64, device=self.dev)
        for c0 in range(0, len(self.V), self.chunk):
            V = self.V[c0:c0 + self.chunk]
            Ec = torch.zeros((len(V), nb, nb), dtype=torch.float64, device=self.dev)
            Fc = torch.zeros((len(V), nb), dtype=torch.float64, device=self.dev)
            h = self._delta(V, co) if co["supg"] else None
            for r, w in self.pts:
                phi, dphi = self._basis(r)
                X, Jinv, det = self._map(V, r)
                g = torch.einsum("ja,cad->cjd", dphi, Jinv)
                b = self._conv(co, X)
                bg = torch.einsum("cd,cjd->cj", b, g)
                test = phi.expand(len(V), nb)
                stab = torch.zeros_like(bg)
                if co["supg"]:
                    s = b.norm(dim=1).clamp_min(1e-300)
                    al = s * h / (2 * co["eps"] * self.p)
                    stab = (h / self.p * (1 / torch.tanh(al) - 1 / al) / (2 * s))[:, None] * bg
                m = (w * det)[:, None]
                Fc += m * (test + stab) * self._source(co, X, b)[:, None]
                if what == "A":
                    left = torch.cat([co["eps"] * g, (test + stab)[:, :, None]], 2)
                    right = torch.cat([g, bg[:, :, None]], 2)
                    Ec.baddbmm_(left * m[:, :, None], right.transpose(1, 2).contiguous())
                else:
                    Ec += (m * (test if what == "M" else stab))[:, :, None] * phi
            E[c0:c0 + self.chunk] = Ec
            rhs.index_add_(0, self.gn[c0:c0 + self.chunk].reshape(-1), Fc.reshape(-1))
        rhs[self.nact:] = 0
        return E, rhs

    def apply(self, E, x, rows=None):
        """The matrix times x; Dirichlet rows are identity rows (rows: their result instead)."""
        y = torch.zeros_like(x)
        step = 1 << 20
        for c0 in range(0, len(E), step):
            gn = self.gn[c0:c0 + step]
            y.index_add_(0, gn.reshape(-1), torch.bmm(E[c0:c0 + step], x[gn][:, :, None]).reshape(-1))
        y[self.nact:] = x[self.nact:] if rows is None else rows
        return y

    def solve(self, E, rhs, x=None, tol=1e-13, restart=150, most=40):
        """GMRES with the diagonal as preconditioner, orthogonalised twice; None if it does not get there."""
        d = torch.zeros_like(rhs)
        d.index_add_(0, self.gn.reshape(-1), torch.diagonal(E, dim1=1, dim2=2).reshape(-1))
        d[self.nact:] = 1
        x = torch.zeros_like(rhs) if x is None else x.clone()
        x[self.nact:] = rhs[self.nact:]
        stop = tol * float((rhs - self.apply(E, x)).norm())
        last = math.inf
        for _ in range(most):
            r = rhs - self.apply(E, x)
            beta = float(r.norm())
            if beta <= stop or beta > 0.5 * last:
                break
            last = beta
            V = torch.empty((restart + 1, len(rhs)), dtype=torch.float64, device=self.dev)
            H = np.zeros((restart + 1, restart))
            V[0] = r / beta
            for k in range(restart):
                w = self.apply(E, V[k] / d)
                h = V[:k + 1] @ w
                w = w - h @ V[:k + 1]
                h2 = V[:k + 1] @ w
                w = w - h2 @ V[:k + 1]
                nw = w.norm()
                V[k + 1] = w / nw
                H[:k + 2, k] = torch.cat([h + h2, nw[None]]).cpu().numpy()
                if (k + 1) % 10 == 0 or k + 1 == restart:
                    e = np.zeros(k + 2)
                    e[0] = beta
                    y, *_ = np.linalg.lstsq(H[:k + 2, :k + 1], e, rcond=None)
                    if np.linalg.norm(H[:k + 2, :k + 1] @ y - e) <= 0.5 * stop:
                        break
            x = x + torch.from_numpy(y).to(self.dev) @ V[:len(y)] / d
        return x if beta <= max(20 * stop, 1e-12 * float(rhs.norm())) else None




def _exact_solve(F, co):
    E, rhs = F.matrices(co, "A")
    x = F.solve(E, rhs)
    return None if x is None else x.cpu().numpy()


def exact(case, seed):
    rng = _rng(seed)
    kind = case["kind"]
    if kind in ("batch", "serve"):
        if kind == "batch":
            meshes = [(1, m, case["levels"]) for m in _batch_m(case)]
        else:
            meshes = _serve_meshes(case)
        return [_exact_solve(_levels_fem(o, m, lv), co) for (o, m, lv), co in zip(meshes, _many_coeffs(len(meshes), rng))]
    n = case["order"] * (case["m"] << (case["k0"] + case["levels"] - 1))
    if n > 130:
        return None  # over 20 seconds
    kw = dict(vertices=_vertices(case["m"], rng)) if kind == "hex" else {}
    P = _problem(case, **kw)
    l = P.levels - 1
    F = _Fem(case["order"], P.cells(l), P.gn(l), P.info(l)["nact"], "cuda")
    if kind == "tcd":
        co = dict(_tcd_coeffs(case, rng), t=0.0)
        u = torch.from_numpy(_pulse(P, co)).to(F.dev)
        P.close()
        return _exact_steps(F, co, u, case["steps"])
    P.close()
    co = _coeffs(case, rng)
    if kind == "matvec":
        E, _ = F.matrices(co, "A")
        return F.apply(E, torch.from_numpy(rng.standard_normal(F.n)).to(F.dev)).cpu().numpy()
    return _exact_solve(F, co)


def _levels_fem(order, m, levels):
    P = pm.Problem(order, m, 0, levels)
    l = levels - 1
    F = _Fem(order, P.cells(l), P.gn(l), P.info(l)["nact"], "cuda")
    P.close()
    return F


def _exact_steps(F, co, u, steps):
    """Crank-Nicolson with the convection matrix at the new time on both sides."""
    M, old = F.matrices(co, "M")
    u[F.nact:] = 0
    for _ in range(steps):
        co["t"] += TAU
        A, new = F.matrices(co, "A")
        T = M + F.matrices(co, "K")[0] if co["supg"] else M
        b = F.apply(T - 0.5 * TAU * A, u, rows=0.0) + 0.5 * TAU * (old + new)
        b[F.nact:] = 0
        u = F.solve(T + 0.5 * TAU * A, b, x=u)
        if u is None:
            return None
        old = new
    return u.cpu().numpy()
