"""The work that programs have this library do, as timed cases.

Seven kinds of pass, each through the public entry points of tahoe_amd.api
and tahoe_amd.batch on a context that is set up beforehand (except for the
batches, whose set-up is part of every solve in real use):

  residual    R(u) and ||R||: the convergence test of every Newton iterate
  product     K(u) assembled, then b = K x (GlobalMatrixT::Multx)
  solve       K(u) assembled, then K x = b on device vectors
  newton      one load step of a single problem to convergence
  krylov      the same with the Newton-Krylov solver (restarted GMRES)
  batch       a batch of RVE solves: pack, context set-up, Newton, results
  path        a static load path of several steps with close_step

Every output is a displacement, residual, product or solution in FP64, of a
computation that is converged or short, so that a change of rounding does
not move it.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from tahoe_amd import api, batch, mesh as M, rve

E1 = 1000.0                                     # Young's modulus of the repository's workloads
ELEMENT = {"tl": api.TOTAL_LAGRANGIAN, "q1p0": api.Q1P0}
MATERIAL = {"simo": api.MAT_SIMO_ISOTROPIC, "stvenant": api.MAT_STVENANT}
PRECISION = {"fp64": api.FP64, "mixed": api.MIXED}
PRECOND = {"jacobi": api.PC_JACOBI, "block": api.PC_BLOCK_JACOBI, "amg": api.PC_AMG}


def listed():
    def cube(name, kind, n, **more):
        nx, ny, nz = (n, n, n) if isinstance(n, int) else n
        return {"name": name, "kind": kind, "nx": nx, "ny": ny, "nz": nz, **more}

    return [
        # the smallest call: one residual of an 8^3 cube, where launches,
        # copies and waits count
        cube("residual-tl-8", "residual", 8, element="tl", material="simo"),
        # an ordinary near-incompressible residual on a ragged mesh
        cube("residual-q1p0-88k", "residual", (45, 38, 51), element="q1p0", material="simo"),
        # assembly into the MSR matrix and a Multx, as the GlobalMatrixT
        # interface asks for them, on an ordinary ragged mesh
        cube("product-tl-62k", "product", (33, 40, 47), element="tl", material="simo"),
        # assembly and a linear solve on device vectors, for callers that
        # keep their own Newton loop
        cube("solve-block-21k", "solve", (24, 31, 28), element="tl", material="simo", precond="block"),
        # the 16^3 cube of the reference run: the first of its load steps,
        # plain FP64 with tight PCG
        cube("newton-fp64-16", "newton", 16, element="tl", material="simo", precision="fp64", precond="jacobi",
             rtol=1e-10),
        # an ordinary mixed-precision load step on a ragged mesh
        cube("newton-mixed-118k", "newton", (50, 52, 45), element="tl", material="simo", precision="mixed",
             precond="jacobi", rtol=1e-3),
        # the largest: one Newton load step at 128^3, mixed precision with
        # the multigrid
        cube("newton-mixed-amg-128", "newton", 128, element="tl", material="simo", precision="mixed", precond="amg",
             rtol=1e-3),
        # the same in plain FP64 on a large ragged mesh: residual, stiffness,
        # expansion and the streaming PCG, inexact Newton
        cube("newton-fp64-892k", "newton", (93, 101, 95), element="tl", material="simo", precision="fp64",
             precond="jacobi", rtol=1e-3),
        # one RVE request on its own: the latency of a served solve
        {"name": "rve-one-q1p0-12", "kind": "batch", "element": "q1p0", "count": 1, "lo": 12, "hi": 12},
        # a served mini-batch of the smallest size class
        {"name": "rve-small-tl", "kind": "batch", "element": "tl", "count": 32, "lo": 4, "hi": 8},
        # a slice of the 4096-RVE run: edges log-uniform 4..24
        {"name": "rve-mix-tl", "kind": "batch", "element": "tl", "count": 384, "lo": 4, "hi": 24},
        # a served mini-batch of the largest size class, near-incompressible
        {"name": "rve-large-q1p0", "kind": "batch", "element": "q1p0", "count": 12, "lo": 16, "hi": 28},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["residual", "product", "solve", "newton", "newton", "newton", "krylov", "batch", "batch", "path"])
    if kind == "batch":
        q1p0 = rng.random() < 0.5
        lo, hi = rng.choice([(4, 8), (9, 15), (16, 28)] if q1p0 else [(4, 8), (9, 15), (16, 24), (4, 24)])
        most = {8: 32, 15: 32, 28: 10, 24: 24}[hi] if q1p0 or lo == 16 else {8: 600, 15: 160, 24: 200}[hi]
        return {"kind": "batch", "element": "q1p0" if q1p0 else "tl", "count": _logint(rng, 1, most), "lo": lo,
                "hi": hi}
    # mesh sizes: element counts log-uniform, edges apart by up to a half
    top = {"residual": 1 << 21, "product": 400000, "solve": 80000, "newton": 600000, "krylov": 600,
           "path": 20000}[kind]
    n = _logint(rng, 64, top)
    a, b = rng.uniform(0.8, 1.25), rng.uniform(0.8, 1.25)
    e = n ** (1.0 / 3.0)
    nx, ny = max(2, round(e * a)), max(2, round(e * b))
    nz = max(2, min(round(n / (nx * ny)), 160))
    case = {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "element": "tl", "material": "simo"}
    if kind == "residual":
        case["element"] = rng.choice(["tl", "q1p0"])
    if kind in ("residual", "product", "solve"):
        case["material"] = rng.choice(["simo", "simo", "stvenant"])
    if kind == "solve":
        case["precond"] = rng.choice(["jacobi", "block"])
    if kind in ("newton", "path"):
        case["precision"] = rng.choice(["fp64", "mixed"])
        case["precond"] = rng.choice(["jacobi", "jacobi", "block"] + (["amg"] if kind == "newton" else []))
        case["rtol"] = 1e-3 if n > 40000 else rng.choice([1e-3, 1e-10])
        if n <= 8000:
            case["element"] = rng.choice(["tl", "q1p0"])
    if kind == "krylov":
        case["precision"], case["precond"], case["rtol"] = "fp64", "jacobi", 1e-3
    return case


# ---- inputs ------------------------------------------------------------------

def _edges(case):
    """Edge lengths of a batch: log-uniform, the same for every seed, so
    that every state of a case is the same amount of work."""
    if case["lo"] == case["hi"]:
        return [case["lo"]] * case["count"]
    return [int(n) for n in rve.log_uniform_edges(case["count"], case["lo"], case["hi"], 4242 + case["count"])]


def _requests(case, seed):
    q1p0 = case["element"] == "q1p0"
    return [rve.Request(i, n, ELEMENT[case["element"]], 0.499 if q1p0 else 0.3, seed * 100003 + i, isochoric=q1p0)
            for i, n in enumerate(_edges(case))]


def _nu(case):
    """Near-incompressible for the Q1P0 residuals (the RVE requests carry
    their own); 0.3 for the load steps, as in the reference's Q1P0 runs."""
    return 0.499 if case["element"] == "q1p0" and case["kind"] == "residual" else 0.3


def _stretch(case):
    """Raise of the top face in one load step, relative to the height: 1 %
    (the 16^3 run's step), less on fine meshes, whose top element layer
    takes the whole raise in the first correction."""
    return min(0.01, (0.08 if _nu(case) > 0.4 else 0.64) / case["nz"])


def _state_field(case, m, seed):
    """A displacement in mid-solve: the affine stretch plus a perturbation
    of up to 2 % of the element size at the free nodes."""
    r = np.random.default_rng([seed, 1])
    h = 1.0 / max(m.shape)
    u = r.uniform(-0.02 * h, 0.02 * h, (m.nnd, 3))
    if _nu(case) > 0.4:
        u *= 0.05               # near-incompressible: small volume changes
    s = _stretch(case)
    u[:, 2] += s * m.X[:, 2]
    u[:, :2] -= 0.5 * s * m.X[:, :2]
    return u


def _mesh(case, seed):
    """The perturbed unit cube, its kinematic cards (bottom fixed, top
    raised) and the (node, dof) pairs without a card."""
    m = M.cube(0, seed=seed, nxyz=(case["nx"], case["ny"], case["nz"]))
    kbc = M.kbc_uniaxial(m, _stretch(case))
    free = np.ones((m.nnd, 3), dtype=bool)
    free[kbc.nodes, kbc.dofs] = False
    return m, kbc, free


def _solid(case, m, kbc):
    s = api.Solid(0)
    s.set_mesh(m.X, m.conn, m.mat)
    s.set_material(0, *api.mu_kappa(E1, _nu(case)))
    s.set_formulation(ELEMENT[case["element"]])
    s.set_material_model(MATERIAL[case["material"]])
    s.set_precision(PRECISION[case.get("precision", "fp64")])
    s.set_kbc(kbc.nodes, kbc.dofs, kbc.values)
    s.set_preconditioner(PRECOND[case.get("precond", "jacobi")])
    if case["kind"] == "krylov":
        s.set_linear_solver(api.LIN_GMRES, 100)
    s.initialize()
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        problems = [q.problem() for q in _requests(case, seed)]
        return {"case": case, "problems": problems, "solid": api.Solid(0), "opts": api.Solid.opts(lin_rtol=1e-3)}
    m, kbc, free = _mesh(case, seed)
    s = _solid(case, m, kbc)
    st = {"case": case, "solid": s}
    if kind in ("residual", "product", "solve"):
        s.set_displacement(_state_field(case, m, seed))
    if kind == "product":
        st["x"] = np.random.default_rng([seed, 2]).standard_normal(s.n_eq)
    if kind == "solve":
        st["b"] = torch.from_numpy(np.random.default_rng([seed, 3]).standard_normal(s.n_eq)).cuda()
        st["x"] = torch.empty_like(st["b"])
    if kind in ("newton", "krylov", "path"):
        # a digit more than the default: on ill-conditioned meshes the
        # displacement is a digit less accurate than the residual
        st["opts"] = s.opts(rel_tol=1e-11, lin_rtol=case["rtol"], lin_maxit=0 if kind == "krylov" else 200000)
    if kind == "path":
        st["u0"] = np.zeros((m.nnd, 3))
    return st


# ---- one pass ----------------------------------------------------------------

def run(state):
    case, s = state["case"], state["solid"]
    kind = case["kind"]
    if kind == "residual":
        R, norm = s.form_rhs()
        return {"R": R, "norm": norm}
    if kind == "product":
        s.form_lhs()
        return s.multx(state["x"])
    if kind == "solve":
        s.form_lhs()
        s.solve_noalloc(state["b"].data_ptr(), state["x"].data_ptr())
        return state["x"]
    if kind == "batch":
        pk = batch.pack(state["problems"])
        q1p0 = case["element"] == "q1p0"
        batch.configure(s, pk, formulation=ELEMENT[case["element"]], precision=api.MIXED,
                        precond=api.PC_BLOCK_JACOBI if q1p0 else api.PC_JACOBI)
        us, _ = batch.solve_one_step_partial(s, pk, state["opts"])
        return [np.concatenate([u if u is not None else np.full_like(p.mesh.X, np.nan)
                                for u, p in zip(us, state["problems"])])]
    if kind == "path":
        s.set_displacement(state["u0"])
        s.close_step()
        us, _ = api.static_solve(s, 3, state["opts"])
        return us
    # newton, krylov: from the last converged state (zero)
    s.reset_step()
    s.apply_kbc(1.0)
    s.newton(state["opts"])
    return s.displacement()


# ---- the work of one pass ----------------------------------------------------

def _counts(case):
    if case["kind"] == "batch":
        e = _edges(case)
        return sum(n ** 3 for n in e), sum((n + 1) ** 3 for n in e), max(e)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    return nx * ny * nz, (nx + 1) * (ny + 1) * (nz + 1), max(nx, ny, nz)


# operations per element: a residual (8 points x kinematics, stress, B^T s),
# the upper triangle of a stiffness (36 node blocks x 8 points x 99
# multiply-adds); a Q1P0 stiffness is 25 residuals
RES_FLOPS, STIFF_FLOPS = 6.2e3, 57e3


def work(case):
    """One pass's mesh and vectors read and written once, and for each
    tangent and each inner iteration the upper half of the operator once
    (14 of a node's 27 blocks, 9 values each); the iteration counts are the
    usual growth with the edge (Jacobi about 1.5 iterations per element of
    edge and decade of the tolerance, multigrid about 14 per decade-third)."""
    nel, nnd, edge = _counts(case)
    mesh_b = 36.0 * nel + 72.0 * nnd
    val = 4.0 if case["kind"] == "batch" or case.get("precision") == "mixed" else 8.0
    op_b, op_f = 14 * 9 * val * nnd, 27 * 18.0 * nnd
    q1p0 = case.get("element") == "q1p0"
    res_f = RES_FLOPS * nel
    stiff_f = 25 * RES_FLOPS * nel if q1p0 else STIFF_FLOPS * nel
    kind = case["kind"]
    if kind == "residual":
        return {"bytes": mesh_b, "flops": res_f}
    if kind == "product":
        return {"bytes": mesh_b + op_b, "flops": stiff_f + op_f}
    rtol = 1e-12 if kind == "solve" else case.get("rtol", 1e-3)
    its = 1.5 * edge * -math.log10(rtol) / (2.0 if kind == "batch" else 1.0) * (2.0 if q1p0 else 1.0)
    if case.get("precond") == "amg":
        its = 14.0 * -math.log10(rtol) / 3.0
    tangents = {"solve": 1, "newton": 5, "krylov": 5, "path": 12, "batch": 4}[kind]
    return {"bytes": tangents * (mesh_b + (1 + its) * (op_b + 120.0 * nnd)),
            "flops": tangents * (res_f + stiff_f + its * op_f)}


# ---- the same in plain torch, in 64 bits --------------------------------------

_SIGNS = [[-1, -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1], [-1, -1, 1], [1, -1, 1], [1, 1, 1], [-1, 1, 1]]


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _inverse(a):
    """Determinant and inverse of [..., 3, 3] by cofactors."""
    r0, r1, r2 = a.unbind(-2)
    c = torch.stack([torch.linalg.cross(r1, r2), torch.linalg.cross(r2, r0), torch.linalg.cross(r0, r1)], -1)
    det = (r0 * c[..., 0]).sum(-1)
    return det, c / det[..., None, None]


def _force(X, u, mu, kappa, element, material):
    """Internal force [e, 8, 3] of hexahedra with nodes X and displacements
    u [e, 8, 3], moduli [e], 2x2x2 Gauss points."""
    sg = torch.tensor(_SIGNS, dtype=torch.float64, device=X.device)
    p = sg / math.sqrt(3.0)
    one = 1.0 + sg[None, :, :] * p[:, None, :]                                     # [q, a, 3]
    d = 0.125 * sg[None] * torch.stack([one[..., 1] * one[..., 2], one[..., 0] * one[..., 2],
                                        one[..., 0] * one[..., 1]], -1)            # dN_a/dxi_k at q
    eye = torch.eye(3, dtype=torch.float64, device=X.device)
    det0, inv0 = _inverse(torch.einsum("eai,qak->eqik", X, d))
    g0 = torch.einsum("qak,eqkl->eqal", d, inv0)                                   # dN/dX
    F = eye + torch.einsum("eai,eqal->eqil", u, g0)
    J, Fi = _inverse(F)
    mu, kappa = mu[:, None, None, None], kappa[:, None, None, None]
    if element == "q1p0":
        detc, _ = _inverse(torch.einsum("eai,qak->eqik", X + u, d))
        H, v = det0.sum(1, keepdim=True), detc.sum(1, keepdim=True)
        F = (v / (H * J)).pow(1.0 / 3.0)[..., None, None] * F
        Jb = (v / H)[..., None, None]
    else:
        Jb = J[..., None, None]
    b = F @ F.transpose(-1, -2)
    if material == "stvenant":
        lam = kappa - 2.0 * mu / 3.0
        tr = 0.5 * (b.diagonal(dim1=-2, dim2=-1).sum(-1)[..., None, None] - 3.0)
        tau = lam * tr * b + mu * (b @ b - b)
    else:
        bb = Jb.pow(-2.0 / 3.0) * b
        mean = bb.diagonal(dim1=-2, dim2=-1).sum(-1)[..., None, None] / 3.0
        tau = mu * (bb - mean * eye) + 0.5 * kappa * (Jb * Jb - 1.0) * eye
    g = torch.einsum("eqal,eqlj->eqaj", g0, Fi)                                    # dN/dx
    if element != "q1p0":
        return torch.einsum("eq,eqij,eqaj->eai", det0, tau, g)
    # mean dilatation: the pressure part acts on the element's mean gradient
    w = detc                                                                       # det0 J
    mean_g = torch.einsum("eq,eqaj->eaj", w / v, g)
    sig = tau / Jb * (Jb[..., 0, 0] / J)[..., None, None]
    press = sig.diagonal(dim1=-2, dim2=-1).sum(-1) / 3.0
    return torch.einsum("eq,eqij,eqaj->eai", w, sig, g) + \
        torch.einsum("eq,eqaj->eaj", w * press, mean_g[:, None] - g)


class _Reference:
    """Residual, tangent and solve of one mesh in torch, FP64."""

    CHUNK = 1 << 17

    def __init__(self, X, conn, mu, kappa, free, element, material="simo"):
        dev = _device()
        put = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
        self.conn = put(conn).long()
        self.X, self.mu, self.kappa = put(X), put(mu), put(kappa)
        self.free = put(free).double()
        self.element, self.material = element, material

    def _chunks(self):
        n = self.conn.shape[0]
        return [slice(b, min(b + self.CHUNK, n)) for b in range(0, n, self.CHUNK)]

    def _force(self, s, ue):
        return _force(self.X[self.conn[s]], ue, self.mu[s], self.kappa[s], self.element, self.material)

    def residual(self, u):
        R = torch.zeros_like(u)
        for s in self._chunks():
            f = self._force(s, u[self.conn[s]])
            R.index_add_(0, self.conn[s].reshape(-1), -f.reshape(-1, 3))
        return R * self.free

    def tangent(self, u):
        """Element tangents [e, 24, 24] (symmetric part) and 1/diag."""
        n = self.conn.shape[0]
        self.K = torch.empty((n, 24, 24), dtype=torch.float64, device=u.device)
        for s in self._chunks():
            ue = u[self.conn[s]]
            for k in range(24):
                t = torch.zeros_like(ue)
                t[:, k // 3, k % 3] = 1.0
                self.K[s, :, k] = torch.func.jvp(lambda v: self._force(s, v), (ue,), (t,))[1].reshape(-1, 24)
            self.K[s] = 0.5 * (self.K[s] + self.K[s].transpose(1, 2).clone())
        d = torch.zeros_like(u)
        d.index_add_(0, self.conn.reshape(-1), self.K.diagonal(dim1=1, dim2=2).reshape(-1, 3))
        self.dinv = torch.where((self.free > 0) & (d != 0), 1.0 / torch.where(d != 0, d, torch.ones_like(d)),
                                torch.zeros_like(d))

    def apply(self, p):
        y = torch.zeros_like(p)
        for s in self._chunks():
            q = torch.matmul(self.K[s], p[self.conn[s]].reshape(-1, 24, 1))
            y.index_add_(0, self.conn[s].reshape(-1), q.reshape(-1, 3))
        return y * self.free

    def pcg(self, b, rtol, maxit=20000):
        x, r = torch.zeros_like(b), b.clone()
        z = self.dinv * r
        p, rz, bb = z.clone(), (r * z).sum(), float((b * b).sum())
        for _ in range(maxit):
            q = self.apply(p)
            alpha = rz / (p * q).sum()
            x += alpha * p
            r -= alpha * q
            if float((r * r).sum()) <= rtol * rtol * bb:
                break
            z = self.dinv * r
            rz, old = (r * z).sum(), rz
            p = z + (rz / old) * p
        return x

    def newton(self, u, tol=1e-12, rtol=1e-4):
        first = last = None
        for _ in range(25):
            R = self.residual(u)
            n = float(R.norm())
            first, last = (n, n) if first is None else (first, last)
            # done, or at the rounding of the residual itself
            if n <= tol * first or (n <= 1e-9 * first and n > 0.1 * last):
                break
            last = n
            self.tangent(u)
            u = u + self.pcg(R, rtol)
        return u


def _moduli(nel, mat, E, nu):
    mk = np.array([api.mu_kappa(e, n) for e, n in zip(E, nu)])
    return mk[mat, 0], mk[mat, 1]


def exact(case, seed):
    kind = case["kind"]
    nel, _, edge = _counts(case)
    if kind == "batch":
        if nel > (30000 if case["element"] == "q1p0" else 1200000):
            return None
        pk = batch.pack([q.problem() for q in _requests(case, seed)])
        mu, kappa = _moduli(len(pk.conn), pk.mat, *zip(*pk.materials))
        free = np.ones((len(pk.X), 3), dtype=bool)
        free[pk.kbc.nodes, pk.kbc.dofs] = False
        ref = _Reference(pk.X, pk.conn, mu, kappa, free, case["element"])
        u = pk.u0.copy()
        u[pk.kbc.nodes, pk.kbc.dofs] = pk.kbc.values
        u = ref.newton(torch.from_numpy(u).to(_device())).cpu().numpy()
        return [np.concatenate([u[b:b + n] for b, n in zip(pk.node_begin[:-1], pk.node_count)])]
    if kind in ("newton", "krylov", "path") and nel > (30000 if case["element"] == "q1p0" else 300000):
        return None
    m, kbc, free = _mesh(case, seed)
    mu, kappa = _moduli(m.nel, m.mat, [E1], [_nu(case)])
    ref = _Reference(m.X, m.conn, mu, kappa, free, case["element"], case["material"])
    act = torch.from_numpy(free).to(_device())
    put = lambda a: torch.from_numpy(a).to(_device())  # noqa: E731
    if kind in ("residual", "product", "solve"):
        u = put(_state_field(case, m, seed))
        if kind == "residual":
            R = ref.residual(u)[act]
            return {"R": R, "norm": float(R.norm())}
        ref.tangent(u)
        v = torch.zeros_like(u)
        if kind == "product":
            v[act] = put(np.random.default_rng([seed, 2]).standard_normal(int(free.sum())))
            return ref.apply(v)[act]
        v[act] = put(np.random.default_rng([seed, 3]).standard_normal(int(free.sum())))
        return ref.pcg(v, 1e-14)[act]
    u = torch.zeros((m.nnd, 3), dtype=torch.float64, device=_device())

    def load(u, t):
        u = u.clone()
        u[put(kbc.nodes).long(), put(kbc.dofs).long()] = t * put(kbc.values)
        return u

    if kind == "path":
        steps = []
        for k in (1, 2, 3):
            u = ref.newton(load(u, k / 3.0))
            steps.append(u)
        return torch.stack(steps)
    return ref.newton(load(u, 1.0))
