"""Performance cases: what a program built on this package has it do, through the
public entry points, over the sizes, geometries, physics and precisions that
the tests, the scenarios and the benchmark of this repository use.

  listed()            the named cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) the context, state and buffers a program holds before the call
  run(state)          one pass; its outputs
  work(case)          bytes and operations no implementation can do without
  exact(case, seed)   the outputs in 64 bits from plain torch (None where that has no
                      value or takes too long)

Operations (``op``):
  assemble  one residual and one tangent on a new iterate (the two callbacks of
            a Newton iteration), device vectors in and out
  residual  the residual alone (a line-search trial)
  tangent   the tangent alone (a Newton refresh, a multigrid level)
  loadstep  one load step: Newton, line search, GMRES and preconditioner
  net       loss and gradients of the warm-start network on one training pair
"""
import math

import numpy as np
import torch

import igap4_amd as ig
from igap4_amd import _lib
from igap4_amd.assm import default_solver_opts
from igap4_amd.loadstep import run_load_steps
from igap4_amd.warmstart import WarmStartNet

DT = 1e-3          # time step of the transient workload


def _case(name, op, nel, phys="static", geom="beam", prec="f64", pc="f64"):
    c = {"op": op, "nx": nel[0], "ny": nel[1], "nz": nel[2], "phys": phys, "geom": geom, "prec": prec, "pc": pc}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest patch of the tests and the warm-start ablation: both callbacks are a few launches each
        _case("assemble 16x4x4 f64", "assemble", (16, 4, 4)),
        # the load-step workload's patch: a line-search trial, and a Newton refresh
        _case("residual 64x16x16", "residual", (64, 16, 16)),
        _case("tangent 64x16x16 f64", "tangent", (64, 16, 16)),
        # the benchmark's step: the largest single-GPU patch
        _case("assemble 256x64x64 f64", "assemble", (256, 64, 64)),
        # the FP32 tangent (preconditioner levels, inexact Newton) on the 256k-element patch
        _case("tangent 160x40x40 f32", "tangent", (160, 40, 40), prec="f32"),
        # igabeamtest's distorted geometry with the reference's three-well energy
        _case("assemble perturbed 64x16x16 f64", "assemble", (64, 16, 16), phys="static-ref", geom="perturbed"),
        # a rational patch of odd element counts, FP32 tangent
        _case("assemble nurbs 45x23x17 f32", "assemble", (45, 23, 17), phys="static-ref", geom="nurbs", prec="f32"),
        # the transient workload: an iteration of a time step with the FP32 tangent
        _case("assemble transient 128x32x32 f32", "assemble", (128, 32, 32), phys="transient", prec="f32"),
        # the periodic cube of the reference's example, refined, FP64
        _case("assemble transient periodic 24x24x24 f64", "assemble", (24, 24, 24), phys="transient", geom="periodic"),
        # one load step of the ramp from the previous solution, multigrid, everything FP64
        _case("loadstep 64x16x16 f64", "loadstep", (64, 16, 16)),
        # the same with FP32 multigrid levels smoothing with 16-bit matrices
        _case("loadstep 128x32x32 mixed", "loadstep", (128, 32, 32), pc="mixed"),
        # the warm-start network on the 64x16x16 patch's control-point grid: one training pair
        _case("net 66x18x18", "net", (66, 18, 18)),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["assemble", "assemble", "residual", "tangent", "tangent", "loadstep", "net"])
    if op == "loadstep":
        # the beam's 4:1:1 element counts; directions that the multigrid can halve
        m = rng.choice([8, 12, 16, 20, 24])
        return _case(None, op, (4 * m, m, rng.choice([m, m - 4])), pc=rng.choice(["f64", "mixed"]))
    if op == "net":
        m = _spread(rng, 6, 24)
        return _case(None, op, (_spread(rng, 12, 80), m + rng.randrange(3), m))
    geom = rng.choice(["beam", "beam", "periodic", "perturbed", "nurbs"])
    phys = rng.choice(["static", "static-ref", "transient"])
    big = 150000 if geom in ("beam", "periodic") else 40000
    while True:
        nel = (_spread(rng, 5, 160), _spread(rng, 5, 48), _spread(rng, 5, 48))
        if 200 <= nel[0] * nel[1] * nel[2] <= (big if phys != "transient" else big // 2):
            break
    return _case(None, op, nel, phys=phys, geom=geom, prec=rng.choice(["f64", "f32"]))


# ------------------------------------------------------------------ inputs
def _mesh(c):
    nel = (c["nx"], c["ny"], c["nz"])
    per = (1, 1, 1) if c["geom"] == "periodic" else (0, 0, 0)
    mesh = ig.MeshIGABeam(L=(1, 1, 1) if c["geom"] == "periodic" else (4, 1, 1), nelem=nel, periodic=per,
                          perturbed=c["geom"] == "perturbed")
    if c["geom"] == "nurbs":
        x = mesh.X.reshape(-1, 3)
        mesh.w[:] = 1.0 + 0.2 * np.sin(1.3 * x[:, 0]) * np.cos(2.1 * x[:, 1] + 0.7 * x[:, 2])
    return mesh


def _par(c):
    """(kind, par_mat, energy coefficients or None)"""
    if c["phys"] == "transient":
        par = [0.25, 0.50, 500., 250., 0.025, 1.0, 1.0, DT, 0.0]
        return "transient", par, None
    return "static", None, (ig.SVK_COEF if c["phys"] == "static" else None)


def _tip(seed):
    return 0.05 * (1.0 + 0.2 * math.sin(1.0 + 0.37 * seed))


def _bc(c, seed):
    if c["phys"] == "transient" or c["geom"] == "periodic":
        return ig.BCDefault()
    return ig.BCClampedTip(tip=_tip(seed))


def _state(mesh, c, seed):
    """Smooth displacements of the owned control points (levels x ndof): a few
    long waves with seeded directions and phases, amplitude 0.01 of a width."""
    rng = np.random.default_rng(seed)
    na, nb = mesh.na, mesh.nb
    X = torch.from_numpy(np.ascontiguousarray(mesh.X.reshape(na + (3,))[:nb[0], :nb[1], :nb[2]])).cuda().reshape(-1, 3)
    L = torch.tensor(mesh.L, dtype=torch.float64, device="cuda")
    step = 2 if c["geom"] == "periodic" else 1   # whole periods on the periodic cube
    out = []
    for amp in (0.01, 0.01 * DT, 0.01 * DT):
        f = torch.zeros_like(X)
        for _ in range(4):
            k = torch.tensor(rng.integers(1, 3, 3) * step, dtype=torch.float64, device="cuda")
            d = torch.tensor(rng.standard_normal(3), device="cuda")
            f += torch.outer(torch.sin(math.pi * ((X / L) @ k) + rng.uniform(0, 2 * math.pi)), amp * d / d.norm())
        out.append(f.reshape(-1))
    if c["phys"] != "transient":
        return out[0]
    # current iterate, previous level, the one before: increments of a time step
    u1 = out[0]
    return torch.cat([u1 + out[1], u1, u1 - out[2]])


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = case
    if case["op"] == "net":
        grid = (case["nx"], case["ny"], case["nz"])
        s.net = WarmStartNet(grid, seed=0)
        s.params, s.x, s.target = _net_inputs(case, seed)
        s.net.set_params(s.params)
        return s
    mesh = _mesh(case)
    if case["op"] == "loadstep":
        s.tip = _tip(seed)
        s.A = ig.Assm(mesh, ig.PhysGradElast(coef=ig.SVK_COEF), ig.BCClampedTip(tip=0.0), device=0)
        s.U0 = np.zeros(s.A.ndof)
        # linear solves to 1e-8, as in the precision study: with the default 1e-5 the
        # displacements of a step are only determined to about 1e-9
        s.opts = default_solver_opts(pc="mg", pc_order=1, pc_lag=4, ksp_rtol=1e-8,
                                     pc_fp32=2 if case["pc"] == "mixed" else 0)
        return s
    kind, par, coef = _par(case)
    phys = ig.PhysGradElastTime(par=par) if kind == "transient" else ig.PhysGradElast(coef=coef)
    s.A = ig.Assm(mesh, phys, _bc(case, seed), device=0)
    n = s.A.ndof
    H = _state(mesh, case, seed)
    s.A.set_uhist(H.cpu().numpy())
    s.U = H[:n].clone()
    s.prec = _lib.IGAP_F64 if case["prec"] == "f64" else _lib.IGAP_F32
    s.R = torch.empty(n, dtype=torch.float64, device="cuda") if case["op"] != "tangent" else None
    s.vals = None
    if case["op"] != "residual":
        s.vals = torch.empty(s.A.nnz, dtype=torch.float64 if case["prec"] == "f64" else torch.float32, device="cuda")
    return s


def run(s):
    op = s.case["op"]
    if op == "net":
        loss, g = s.net.gradients(s.x, s.target)
        return {"loss": np.float32(loss), "grad": g}
    if op == "loadstep":
        hist = []
        run_load_steps(s.A, 20, tip_total=s.tip, guess="previous", opts=s.opts, history=hist, start=1, max_steps=1,
                       prev=[s.U0], start_rtol=1e-10)
        return {"U": hist[0]}
    out = {}
    if s.R is not None:
        s.A.residual_dev(s.U.data_ptr(), s.R.data_ptr())
        out["R"] = s.R
    if s.vals is not None:
        s.A.tangent_dev(s.U.data_ptr(), s.vals.data_ptr(), s.prec)
        out["K"] = s.vals
    return out


# ------------------------------------------------------------------ work
def _nnz(c):
    """9 x the number of coupled control-point pairs"""
    n = 9
    for d in ("nx", "ny", "nz"):
        m = c[d]
        n *= 5 * m if c["geom"] == "periodic" else 5 * (m + 2) - 6
    return n


def work(case):
    c = case
    if c["op"] == "net":
        v = c["nx"] * c["ny"] * c["nz"]
        # four layers forward, four weight gradients, three input gradients
        return {"bytes": 4 * v * (9 + 3) + 2 * 4 * 4 * 27 * 256, "flops": 11 * 2 * 27 * 256 * v}
    nel = c["nx"] * c["ny"] * c["nz"]
    per = c["geom"] == "periodic"
    ncp = nel if per else (c["nx"] + 2) * (c["ny"] + 2) * (c["nz"] + 2)
    levels = 3 if c["phys"] == "transient" else 1
    vec = 8 * 3 * ncp
    # sum-factorised fields, pointwise stresses and projection of 64 points
    r = {"bytes": vec * (levels + 2) + 8 * ncp, "flops": nel * (2 * 3 * 2400 * levels + 64 * 600)}
    # pointwise tangents of 64 points and their sum-factorised contraction
    k = {"bytes": vec * (levels + 1) + 8 * ncp + _nnz(c) * (8 if c["prec"] == "f64" else 4), "flops": nel * 700000}
    if c["op"] == "residual":
        return r
    if c["op"] == "tangent":
        return k
    if c["op"] == "assemble":
        return {"bytes": r["bytes"] + k["bytes"], "flops": r["flops"] + k["flops"]}
    # a load step: at least three Newton iterations (residual, tangent) of six
    # Krylov iterations, each with the operator and two finest-level smoothing
    # sweeps of three products
    low = 20 / 9 if c["pc"] == "mixed" else 8
    return {"bytes": 3 * (r["bytes"] + k["bytes"]) + 18 * _nnz(c) * (8 + 6 * low),
            "flops": 3 * (r["flops"] + k["flops"]) + 18 * 7 * 2 * _nnz(c)}


# ------------------------------------------------------------------ 64 bits
def _net_inputs(c, seed):
    """Parameters of a network part way through training (every layer nonzero)
    and one training pair: unit-scale increments, their second differences and
    the load increment on the end face; a smooth target."""
    g = torch.Generator().manual_seed(int(seed))
    shape = (c["nx"], c["ny"], c["nz"])
    V = shape[0] * shape[1] * shape[2]
    P = torch.zeros(4, 27 * 256 + 16)
    for l in range(4):
        ci, co = (9 if l == 0 else 16), (3 if l == 3 else 16)
        W = torch.zeros(27, 16, 16)
        W[:, :co, :ci] = (2 * torch.rand(27, co, ci, generator=g) - 1) * math.sqrt(6.0 / (27 * ci))
        b = torch.zeros(16)
        b[:co] = 0.05 * torch.randn(co, generator=g)
        P[l] = torch.cat([W.reshape(-1), b])
    ax = [torch.linspace(0, 1, n) for n in shape]
    grid = torch.stack(torch.meshgrid(*ax, indexing="ij"), -1).reshape(V, 3)
    k = math.pi * (1 + 3 * torch.rand(3, 9, generator=g))
    x = torch.sin(grid @ k + 6.3 * torch.rand(9, generator=g)) + 0.02 * torch.randn(V, 9, generator=g)
    x[:, 6:] *= (grid[:, :1] == 1).float()
    t = torch.cos(grid @ k[:, :3]) + 0.1 * torch.randn(V, 3, generator=g)
    return P.reshape(-1).numpy(), x.numpy(), t.numpy()


def _exact_net(c, seed):
    P, x, t = (torch.from_numpy(a).double() for a in _net_inputs(c, seed))
    shape = (c["nx"], c["ny"], c["nz"])
    P = P.reshape(4, -1)
    Ws = [P[l, :27 * 256].reshape(27, 16, 16).clone().requires_grad_() for l in range(4)]
    bs = [P[l, 27 * 256:].clone().requires_grad_() for l in range(4)]
    a = torch.zeros(shape + (16,), dtype=torch.float64)
    a[..., :9] = x.reshape(shape + (9,))
    for l, dil in enumerate((1, 2, 4, 1)):
        pad = torch.nn.functional.pad(a, (0, 0, dil, dil, dil, dil, dil, dil))
        z = bs[l]
        for k in range(27):
            o = [dil * (k // 9), dil * ((k // 3) % 3), dil * (k % 3)]
            z = z + pad[o[0]:o[0] + shape[0], o[1]:o[1] + shape[1], o[2]:o[2] + shape[2]] @ Ws[l][k].T
        a = torch.relu(z) if l < 3 else z
    loss = ((a[..., :3].reshape(-1, 3) - t) ** 2).mean()
    loss.backward()
    g = torch.cat([torch.cat([Ws[l].grad.reshape(-1), bs[l].grad]) for l in range(4)])
    return {"loss": np.float64(loss.detach()), "grad": g.numpy()}


def _bspline_tables(kv, nel):
    """[element][Gauss point][order][function] of the quadratic B-splines, and
    weights x span [element][Gauss point]"""
    q, w = np.polynomial.legendre.leggauss(4)
    q, w = 0.5 * (q + 1), 0.5 * w
    t = np.zeros((nel, 4, 3, 3))
    wt = np.zeros((nel, 4))
    for e in range(nel):
        k = kv[e:e + 6]
        x = (1 - q) * k[2] + q * k[3]
        h, a, b = k[3] - k[2], k[3] - k[1], k[4] - k[2]
        t[e, :, 0, 0] = (k[3] - x) ** 2 / (a * h)
        t[e, :, 0, 1] = (x - k[1]) * (k[3] - x) / (a * h) + (k[4] - x) * (x - k[2]) / (b * h)
        t[e, :, 0, 2] = (x - k[2]) ** 2 / (b * h)
        t[e, :, 1, 0] = -2 * (k[3] - x) / (a * h)
        t[e, :, 1, 2] = 2 * (x - k[2]) / (b * h)
        t[e, :, 1, 1] = -t[e, :, 1, 0] - t[e, :, 1, 2]
        t[e, :, 2, 0] = 2 / (a * h)
        t[e, :, 2, 2] = 2 / (b * h)
        t[e, :, 2, 1] = -2 / (a * h) - 2 / (b * h)
        wt[e] = w * h
    return t, wt


_PAIR = [(0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)]


def _jets(T, w, X):
    """Physical jets [e][q][slot][basis] and det G [e][q] from the 1-D tables
    T[d][e][q][order][i], weights w[e][27] and control points X[e][27][3]."""
    E = w.shape[0]

    def prod(ox, oy, oz):
        return torch.einsum("exi,eyj,ezk->exyzijk", T[0][:, :, ox], T[1][:, :, oy], T[2][:, :, oz]).reshape(E, 64, 27)

    N = {(): prod(0, 0, 0)}
    for i in range(3):
        N[(i,)] = prod(*[1 if d == i else 0 for d in range(3)])
    for i, j in _PAIR:
        N[(i, j)] = prod(*[(d == i) + (d == j) for d in range(3)])
    N = {k: v * w[:, None, :] for k, v in N.items()}
    W = {k: v.sum(-1, keepdim=True) for k, v in N.items()}
    R = {(): N[()] / W[()]}
    for i in range(3):
        R[(i,)] = (N[(i,)] - R[()] * W[(i,)]) / W[()]
    for i, j in _PAIR:
        R[(i, j)] = (N[(i, j)] - R[(i,)] * W[(j,)] - R[(j,)] * W[(i,)] - R[()] * W[(i, j)]) / W[()]
    G = torch.stack([torch.einsum("eqb,ebd->eqd", R[(i,)], X) for i in range(3)], -1)    # dx_d / dxi_i
    Gi = torch.linalg.inv(G)                                                              # [i][d]
    D1 = torch.einsum("eqib,eqid->eqdb", torch.stack([R[(i,)] for i in range(3)], 2), Gi)
    H = torch.empty(E, 64, 3, 3, 27, dtype=N[()].dtype, device=N[()].device)
    for i, j in _PAIR:
        x2 = torch.einsum("eqb,ebd->eqd", R[(i, j)], X)
        H[:, :, i, j] = R[(i, j)] - torch.einsum("eqdb,eqd->eqb", D1, x2)
        H[:, :, j, i] = H[:, :, i, j]
    H = torch.einsum("eqid,eqijb,eqjf->eqdfb", Gi, H, Gi)
    return torch.stack([R[()]] + [D1[:, :, d] for d in range(3)] + [H[:, :, i, j] for i, j in _PAIR], 2), torch.linalg.det(G)


def _coef(c):
    kind, par, coef = _par(c)
    if coef is not None:
        return coef
    r, cu, e0, e345, le = par[:5] if par else (0.25, 0.50, 360., 180., 0.05)
    a = 4.0 / 3.0 * r * (1 - cu)
    D = r * r - 2 * r * r * cu - r * a
    return 2 * cu / D, -a / (r * r * D), -1 / (r * r * D), e0, e345, le


def _energy(coef):
    c2, c3, c4, e0, e345, le = coef

    def psi(u):   # u: 27 = [component][3 first, 6 second derivatives]
        u = u.reshape(3, 9)
        F = u[:, :3] + torch.eye(3, dtype=u.dtype, device=u.device)
        idx = [[0, 1, 2], [1, 3, 4], [2, 4, 5]]
        H = u[:, 3:][:, idx]
        C = F.T @ F
        E11, E22, E33 = 0.5 * (C[0, 0] - 1), 0.5 * (C[1, 1] - 1), 0.5 * (C[2, 2] - 1)
        e24 = (E11 + E22 + E33) / math.sqrt(3)
        e25 = (E11 - E22) / math.sqrt(2)
        e26 = (E11 + E22 - 2 * E33) / math.sqrt(6)
        rho = e25 * e25 + e26 * e26
        K = torch.einsum("ki,kij->ij", F, H)      # dE_II / dX_J
        dev = K - K.sum(0, keepdim=True) / 3
        shear = 0.25 * (C[0, 1] ** 2 + C[0, 2] ** 2 + C[1, 2] ** 2)
        return (c3 * e26 * (e26 * e26 - 3 * e25 * e25) + c2 * rho + c4 * rho * rho + e0 * e24 * e24 + e345 * shear
                + le * le * (dev * dev).sum())

    return psi


def _rule():
    """Nodes and weights of the truncated average of a polynomial of degree
    <= 7 along the increment: residual a0 + a1/2 + a2/3 + a3/4, tangent
    (b0/2 + b1/3 + b2/4)/2."""
    s = 2 * np.cos(np.pi * (np.arange(8) + 0.5) / 8)
    V = np.vander(s, 8, increasing=True).T
    return s, np.linalg.solve(V, [1, 1 / 2, 1 / 3, 1 / 4, 0, 0, 0, 0]), np.linalg.solve(V, [1 / 4, 1 / 6, 1 / 8, 0, 0, 0, 0, 0])


def _sorted_stencil(n, periodic, dev):
    """per point of one direction the offsets 0..4 (-2..2) in column order, and
    which of them exist"""
    a = torch.arange(n, device=dev)[:, None] + torch.arange(-2, 3, device=dev)[None]
    if periodic:
        order = torch.argsort(a % n, dim=1)
        return order, torch.ones_like(a, dtype=torch.bool)
    return torch.arange(5, device=dev).expand(n, 5), (a >= 0) & (a < n)


def exact(case, seed):
    c = case
    if c["op"] == "loadstep":
        return None
    if c["op"] == "net":
        return _exact_net(c, seed)
    nel = (c["nx"], c["ny"], c["nz"])
    ne = nel[0] * nel[1] * nel[2]
    if ne > (20000 if c["phys"] == "transient" else 150000):
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    mesh = _mesh(c)
    na, nb = mesh.na, mesh.nb
    kind, par, _ = _par(c)
    H = _state(mesh, c, seed).reshape(-1, nb[0] * nb[1] * nb[2], 3).to(dev)
    X = torch.from_numpy(mesh.X).to(dev).reshape(-1, 3)
    wts = torch.from_numpy(mesh.w).to(dev)
    T, WT = zip(*[_bspline_tables(mesh.knots[d], nel[d]) for d in range(3)])
    T = [torch.from_numpy(t).to(dev) for t in T]
    WT = [torch.from_numpy(t).to(dev) for t in WT]
    psi = _energy(_coef(c))
    grad, hess = torch.func.vmap(torch.func.grad(psi)), torch.func.vmap(torch.func.hessian(psi))
    ncp = nb[0] * nb[1] * nb[2]
    want_r, want_k = c["op"] != "tangent", c["op"] != "residual"
    R = torch.zeros(ncp, 3, dtype=torch.float64, device=dev)
    K = torch.zeros(ncp * 125 if want_k else 1, 9, dtype=torch.float64, device=dev)
    loc = torch.stack(torch.meshgrid(*[torch.arange(3, device=dev)] * 3, indexing="ij"), -1).reshape(27, 3)
    nbt = torch.tensor(nb, device=dev)
    for e0 in range(0, ne, 512):
        e = torch.arange(e0, min(ne, e0 + 512), device=dev)
        E = len(e)
        ed = [e // (nel[1] * nel[2]), (e // nel[2]) % nel[1], e % nel[2]]
        ap = torch.stack(ed, -1)[:, None, :] + loc[None]
        act = (ap[..., 0] * na[1] + ap[..., 1]) * na[2] + ap[..., 2]
        ow = torch.where(ap >= nbt, ap - nbt, ap) if c["geom"] == "periodic" else ap
        own = (ow[..., 0] * nb[1] + ow[..., 1]) * nb[2] + ow[..., 2]
        J, det = _jets([T[d][ed[d]] for d in range(3)], wts[act], X[act])
        wq = torch.einsum("ex,ey,ez->exyz", *[WT[d][ed[d]] for d in range(3)]).reshape(E, 64) * det
        u = torch.einsum("eqab,hebk->heqka", J, H[:, own])
        uj = u[..., 1:].reshape(u.shape[0], E * 64, 27)
        rj = torch.zeros(E, 64, 3, 10, dtype=torch.float64, device=dev)
        Cj = torch.zeros(E, 64, 3, 10, 3, 10, dtype=torch.float64, device=dev)
        if kind == "static":
            rj[..., 1:] = grad(uj[0]).reshape(E, 64, 3, 9)
            if want_k:
                Cj[:, :, :, 1:, :, 1:] = hess(uj[0]).reshape(E, 64, 3, 9, 3, 9)
        else:
            rho, cii = par[5], par[6]
            m0, dd = 0.5 * (uj[1] + uj[2]), 0.5 * (uj[0] - uj[2])
            for s, cr, ct in zip(*_rule()):
                rj[..., 1:] += cr * grad(m0 + s * dd).reshape(E, 64, 3, 9)
                if want_k:
                    Cj[:, :, :, 1:, :, 1:] += ct * hess(m0 + s * dd).reshape(E, 64, 3, 9, 3, 9)
            v = u[..., 0]
            rj[..., 0] = cii * (v[0] - v[2]) / (2 * DT) + rho * (v[0] + v[2] - 2 * v[1]) / DT ** 2
            for k in range(3):
                Cj[:, :, k, 0, k, 0] = cii / (2 * DT) + rho / DT ** 2
        if want_r:
            R.index_add_(0, own.reshape(-1), torch.einsum("eq,eqka,eqab->ebk", wq, rj, J).reshape(-1, 3))
        if want_k:
            CJ = torch.einsum("eqkalm,eqmc->eqkalc", Cj, J)
            Ke = torch.einsum("eqab,eqkalc->ebckl", J * wq[..., None, None], CJ)
            off = ap[:, None, :, :] - ap[:, :, None, :] + 2          # column minus row
            slot = (off[..., 0] * 5 + off[..., 1]) * 5 + off[..., 2]
            K.index_add_(0, (own[:, :, None] * 125 + slot).reshape(-1), Ke.reshape(-1, 9))
    mask = torch.zeros(nb + (3,), dtype=torch.bool, device=dev)
    g = torch.zeros(nb + (3,), dtype=torch.float64, device=dev)
    if c["phys"] != "transient" and c["geom"] != "periodic":
        mask[:2] = True
        mask[-1, :, :, 2] = True
        g[-1, :, :, 2] = _tip(seed)
    mask, g = mask.reshape(ncp, 3), g.reshape(ncp, 3)
    out = {}
    if want_r:
        out["R"] = torch.where(mask, H[0] - g, R).reshape(-1)
    if want_k:
        K = K.reshape(ncp, 125, 3, 3)
        per = c["geom"] == "periodic"
        st = [_sorted_stencil(n, per, dev) for n in nb]
        ii = torch.stack(torch.meshgrid(*[torch.arange(n, device=dev) for n in nb], indexing="ij"), -1).reshape(ncp, 3)
        o = [st[d][0][ii[:, d]] for d in range(3)]
        ok = [st[d][1][ii[:, d]] for d in range(3)]
        slot = ((o[0][:, :, None, None] * 5 + o[1][:, None, :, None]) * 5 + o[2][:, None, None, :]).reshape(ncp, 125)
        ok = (ok[0][:, :, None, None] & ok[1][:, None, :, None] & ok[2][:, None, None, :]).reshape(ncp, 125)
        K = torch.gather(K, 1, slot[:, :, None, None].expand(ncp, 125, 3, 3))
        q = [(ii[:, d][:, None] + o[d] - 2) % nb[d] for d in range(3)]
        col = ((q[0][:, :, None, None] * nb[1] + q[1][:, None, :, None]) * nb[2] + q[2][:, None, None, :]).reshape(ncp, 125)
        dead = mask[:, None, :, None] | mask[col][:, :, None, :]
        one = (col == torch.arange(ncp, device=dev)[:, None])[:, :, None, None] & torch.eye(3, dtype=torch.bool, device=dev)
        K = torch.where(dead, one.double(), K).permute(0, 2, 1, 3)
        out["K"] = K[ok[:, None, :, None].expand(ncp, 3, 125, 3)]
    return out
