"""The measured work of the framework: implicit time steps, whole requests,
coupled steps, groups of systems and solves of a caller's own matrix, each
through the public entry points.

A case is a dict of plain values:
  path       "steps"    time steps of one system that the program keeps
             "request"  a system created, solved and closed (a served request)
             "coupled"  flow step, Gauss-point velocity, heat step
             "group"    one group of systems stepped together
             "crs"      ogsx_solve_crs_noalloc on the caller's device arrays
  mesh       "line", "quad", "hex" or "tet" (cubes of 6 tets); nx, ny, nz cells
  process    "flow", "groundwater" or "heat"
  precision  "fp64" or "ir" (FP32 matrix inside FP64 refinement)
  method     "cg" (symmetric Dirichlet elimination) or "bicgstab" (the
             reference's row-only elimination)
  tensor     anisotropic conductivity tensor per element; gravity: rho g term
  sigma      standard deviation of ln K; steps: time steps of one pass;
  steady     the mass matrix left out
Solves stop at TOL, the tolerance of the reference's own bmskel deck, so that
two correct solvers' solutions agree far more closely than the iterates at a
loose stop would.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import ogs5_amd as ox
from ogs5_amd import mesh as meshes
from ogs5_amd import workloads
from ogs5_amd.fields import lognormal_conductivity
from ogs5_amd.workloads import Scenario, Step

TOL = 1e-12
NPE = {"line": 2, "quad": 4, "hex": 8, "tet": 4}
ROW = {"line": 3, "quad": 9, "hex": 27, "tet": 15}  # entries of an interior row
RHO_G = 1000.0 * 9.81
FLUID_RHO_C = 4.2e6


def _case(path, mesh, nx, ny=0, nz=0, *, process="flow", precision="fp64", method="cg",
          tensor=False, gravity=False, sigma=1.0, steps=1, steady=False, count=1):
    return dict(path=path, mesh=mesh, nx=nx, ny=ny, nz=nz, process=process, precision=precision,
                method=method, tensor=tensor, gravity=gravity, sigma=sigma, steps=steps,
                steady=steady, count=count)


def listed():
    def c(name, *a, **k):
        return dict(_case(*a, **k), name=name)

    return [
        # the smallest call: a 1-D heat column (the reference's bmskel deck is one
        # line element); all latency
        c("line_heat_64", "steps", "line", 64, process="heat", method="bicgstab"),
        # a small served request from creation to solution, on a mesh whose
        # pattern the server holds: what a new system pays
        c("request_quad_75x52", "request", "quad", 75, 52, steps=2),
        # the 2-D confined-aquifer configuration (200 x 200 quads, centre sink)
        c("quad_200x200_fp64", "steps", "quad", 200, 200, steps=2),
        # the same kind of model with the reference's own elimination and solver
        c("quad_173x118_bicgstab", "steps", "quad", 173, 118, process="groundwater",
          method="bicgstab"),
        # a ragged larger 2-D model, strongly heterogeneous, mixed precision
        c("quad_487x301_ir", "steps", "quad", 487, 301, precision="ir", sigma=2.0),
        # 3-D flow with a full permeability tensor and gravity
        c("hex_37x30x23_tensor", "steps", "hex", 37, 30, 23, tensor=True, gravity=True),
        # an ordinary 3-D flow model in plain FP64
        c("hex_85x64x53_fp64", "steps", "hex", 85, 64, 53, sigma=2.0),
        # the 3-D headline configuration: 128^3 hexes, one implicit step
        c("hex_128_ir", "steps", "hex", 128, 128, 128, precision="ir", sigma=2.0),
        # advection-diffusion of heat on tets, one Crank-Nicolson step
        c("tet_heat_80x72x64_ir", "steps", "tet", 80, 72, 64, process="heat", precision="ir",
          method="bicgstab"),
        # pressure-driven flow carrying heat, one coupled step
        c("coupled_tet_36", "coupled", "tet", 36, 36, 36, gravity=True),
        # an ensemble stepped as one group (mixed precision, sides 48 to 192)
        c("group_16_quads_ir", "group", "quad", 48, 192, precision="ir", steps=2, count=16),
        # a caller's own CRS matrix in device memory
        c("crs_quad_230x310_cg", "crs", "quad", 230, 310),
    ]


def draw(rng):
    def side(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    precision = rng.choice(["fp64", "ir"])
    sigma = round(rng.uniform(0.5, 2.0), 2)
    kind = rng.choice(["quad", "quad", "hex", "hex", "heat", "request", "coupled", "group", "crs",
                       "bicgstab"])
    if kind == "quad":
        return _case("steps", "quad", side(24, 600), side(24, 600), precision=precision,
                     sigma=sigma, steps=rng.randint(1, 2), steady=rng.random() < 0.15)
    if kind == "hex":
        return _case("steps", "hex", side(10, 100), side(10, 100), side(10, 100),
                     precision=precision, sigma=sigma, tensor=rng.random() < 0.2,
                     gravity=rng.random() < 0.3)
    if kind == "heat":
        return _case("steps", "tet", side(10, 72), side(10, 72), side(10, 72), process="heat",
                     precision=precision, method="bicgstab", steps=rng.randint(1, 2))
    if kind == "request":
        return _case("request", "quad", side(32, 200), side(32, 200), precision=precision,
                     sigma=sigma, steps=rng.randint(1, 3))
    if kind == "coupled":
        n = side(10, 44)
        return _case("coupled", "tet", n, n, n, precision=precision, gravity=True)
    if kind == "group":
        lo = side(32, 96)
        return _case("group", "quad", lo, side(lo + 8, 220), precision=precision,
                     sigma=sigma, steps=rng.randint(1, 2), count=rng.randint(5, 20))
    if kind == "crs":
        return _case("crs", "quad", side(30, 500), side(30, 500),
                     method=rng.choice(["cg", "bicgstab"]))
    return _case("steps", "quad", side(24, 400), side(24, 400), process="groundwater",
                 precision=precision, method="bicgstab", sigma=sigma)


# ---- inputs ---------------------------------------------------------------
@functools.lru_cache(maxsize=32)
def _mesh(kind, nx, ny, nz):
    if kind == "line":
        return meshes.line_mesh(nx, 10.0)
    if kind == "quad":
        return meshes.quad_mesh(nx, ny, 1000.0, 1000.0 * ny / nx)
    return (meshes.hex_mesh if kind == "hex" else meshes.tet_mesh)(nx, ny, nz)


@functools.lru_cache(maxsize=32)
def _pattern(kind, nx, ny, nz):
    """A program sets a mesh's pattern up once and keeps it (as the serving
    loop does for all requests of one size)."""
    m = _mesh(kind, nx, ny, nz)
    return ox.Pattern(m.n_nodes, m.etype, m.conn)


def _flow(case, m, seed):
    dim = m.dim
    K = lognormal_conductivity(m, math.log(1e-4), case["sigma"], 50.0 if dim == 2 else 8.0,
                               seed, 64)
    stride = 1
    if case["tensor"]:
        # principal axes turned out of the grid, ratio 1 : 0.4 : 0.2
        q = np.linalg.qr(np.random.default_rng(17).standard_normal((dim, dim)))[0]
        t = q @ np.diag([1.0, 0.4, 0.2][:dim]) @ q.T
        K = np.ascontiguousarray((K[:, None] * ((t + t.T) / 2).ravel()[None, :]).ravel())
        stride = dim * dim
    lx = float(m.x.max())
    left, right = m.nodes_where(0, 0.0), m.nodes_where(0, lx)
    idx = np.concatenate([left, right]).astype(np.int64)
    gravity = 0.05 if case["gravity"] else 0.0
    val = np.concatenate([np.full(left.size, 10.0), np.zeros(right.size)])
    centre = m.node_index(*[s // 2 for s in m.shape])
    dt, q = (3600.0, -0.01) if dim == 2 else (100.0, -1e-4)
    process = ox.GROUNDWATER_FLOW if case["process"] == "groundwater" else ox.LIQUID_FLOW
    return Scenario("flow", m, process, np.full(m.n_elem, 1e-4), K, stride, idx, val,
                    np.array([centre], np.int64), np.array([q]), np.zeros(m.n_nodes),
                    [Step(dt, 1.0, steady=case["steady"])] * case["steps"], tol=TOL,
                    rho_g=gravity)


def _heat(case, m, seed):
    rng = np.random.default_rng(seed)
    lam = 2.0
    h = m.h[0]
    vel = None
    if m.dim == 3:
        # one velocity per element (as flow on linear tets gives), curl of a few
        # low modes around a mean along x, grid Peclet numbers 1 to 20
        u = 20.0 * 2.0 * lam / (FLUID_RHO_C * h) / 1.9
        nc, size = m.n_elem // 6, [float(s) for s in m.shape]
        i = np.arange(nc)
        x = (i % m.shape[0] + 0.5) / size[0]
        y = (i // m.shape[0] % m.shape[1] + 0.5) / size[1]
        vx, vy = np.full(nc, 1.0), np.zeros(nc)
        for k in range(1, 4):
            a, ph = rng.uniform(0.1, 0.28), rng.uniform(0.0, 2.0 * math.pi)
            arg = 2.0 * math.pi * (k * x + (4 - k) * y) + ph
            vx += a * np.cos(arg)
            vy -= a * np.cos(arg) * k / (4 - k)
        v = np.stack([vx * u, vy * u, np.zeros(nc)], axis=1)
        vel = np.ascontiguousarray(np.broadcast_to(np.repeat(v, 6, axis=0)[:, :, None],
                                                   (m.n_elem, 3, 5)))
    inlet = m.nodes_where(0, 0.0).astype(np.int64)
    cond = lam * np.exp(0.2 * rng.standard_normal(m.n_elem))
    u0 = 10.0 + rng.uniform(0.0, 2.0, m.n_nodes)
    return Scenario("heat", m, ox.HEAT_TRANSPORT, np.full(m.n_elem, 2.5e6), cond, 1, inlet,
                    np.full(inlet.size, 60.0), np.zeros(0, np.int64), np.zeros(0), u0,
                    [Step(1e5, 0.5)] * case["steps"], tol=TOL,
                    adv_coef=FLUID_RHO_C if vel is not None else 0.0, vel=vel)


def _scenario(case, seed):
    m = _mesh(case["mesh"], case["nx"], case["ny"], case["nz"])
    return (_heat if case["process"] == "heat" else _flow)(case, m, seed)


def _coupled(case, seed):
    flow, heat = workloads.coupled_flow_heat(case["nx"], seed=seed, n_steps=case["steps"])
    flow.tol = heat.tol = TOL
    return flow, heat


def _group(case, seed):
    """count instances, sides spread evenly in the logarithm from nx to ny."""
    r = math.log(case["ny"] / case["nx"]) / max(1, case["count"] - 1)
    out = []
    for i in range(case["count"]):
        s = int(round(case["nx"] * math.exp(r * i)))
        out.append(_scenario(dict(case, nx=s, ny=s), seed * 1000 + i))
    return out


def _crs(case, seed):
    """Five-point conductances of a heterogeneous grid with a storage term, CRS
    with ascending columns; for BiCGStab upwind transport on top (nonsymmetric)."""
    nx, ny = case["nx"], case["ny"]
    rng = np.random.default_rng(seed)
    k = np.exp(rng.standard_normal((ny, nx)))
    ex = 2.0 / (1.0 / k[:, 1:] + 1.0 / k[:, :-1])
    ey = 2.0 / (1.0 / k[1:, :] + 1.0 / k[:-1, :])
    v = 0.5 if case["method"] == "bicgstab" else 0.0
    a = np.zeros((5, ny, nx))  # offsets -nx, -1, 0, 1, nx
    a[0, 1:], a[4, :-1] = -ey, -ey
    a[1, :, 1:], a[3, :, :-1] = -ex - v, -ex
    a[2] = -(a[0] + a[1] + a[3] + a[4]) + 0.02
    off = np.array([-nx, -1, 0, 1, nx])
    have = np.zeros((5, ny, nx), bool)
    have[0, 1:], have[4, :-1], have[1, :, 1:], have[3, :, :-1], have[2] = 1, 1, 1, 1, 1
    have = have.reshape(5, -1).T
    cols = np.arange(nx * ny)[:, None] + off[None, :]
    ptr = np.concatenate([[0], np.cumsum(have.sum(1))])
    b = rng.standard_normal(nx * ny)
    return ptr.astype(np.int32), cols[have].astype(np.int32), a.reshape(5, -1).T[have], b


# ---- the calls ------------------------------------------------------------
def _precision(case):
    return ox.FP32_IR if case["precision"] == "ir" else ox.FP64


def _how(case):
    cg = case["method"] == "cg"
    return dict(method=ox.CG if cg else ox.BICGSTAB,
                dirichlet=ox.DIRICHLET_SYMMETRIC if cg else ox.DIRICHLET_ROW)


def _system(case, sc, kind):
    m = sc.mesh
    pat = _pattern(kind, m.shape[0], m.shape[1] if m.dim > 1 else 0, m.shape[2] if m.dim > 2 else 0)
    s = ox.System(pat, _precision(case))
    s.set_elements(**sc.element_kwargs())
    return pat, s


def prepare(case, seed):
    st = dict(case=case, path=case["path"])
    if case["path"] == "crs":
        ptr, col, val, b = _crs(case, seed)
        dev = [torch.from_numpy(a).cuda() for a in (ptr, col, val, b)]
        st.update(n=b.size, dev=dev, x=torch.zeros(b.size, dtype=torch.float64, device="cuda"))
        return st
    if case["path"] == "coupled":
        flow, heat = _coupled(case, seed)
        pat, sf = _system(case, flow, "tet")
        _, sh = _system(case, heat, "tet")
        st.update(flow=flow, heat=heat, systems=(pat, sf, sh))
        return st
    if case["path"] == "group":
        scs = _group(case, seed)
        g = ox.Group(_precision(case))
        members = []
        for sc in scs:
            s = _system(case, sc, "quad")[1]
            s.set_vector(ox.VEC_IC, sc.u0)
            s.initialize()  # uploads the lists that the group's steps use
            s.assemble(sc.steps[0].dt, sc.steps[0].theta)
            s.add_rhs(sc.st_idx, sc.st_val)
            s.set_dirichlet(sc.bc_idx, sc.bc_val, ox.DIRICHLET_SYMMETRIC)
            g.add(s)
            members.append(s)
        st.update(scs=scs, group=g, members=members)
        return st
    sc = _scenario(case, seed)
    st.update(sc=sc)
    if case["path"] == "request":
        m = sc.mesh
        st.update(pattern=_pattern(case["mesh"], *m.shape, *([0] * (3 - m.dim))))
        return st
    system = _system(case, sc, case["mesh"])
    system[1].set_vector(ox.VEC_IC, sc.u0)
    st.update(system=system)
    return st


def run(st):
    case = st["case"]
    if st["path"] == "steps":
        return workloads.run_gpu(st["sc"], system=st["system"], ic_on_device=True, **_how(case))["x"]
    if st["path"] == "request":
        s = ox.System(st["pattern"], _precision(case))
        s.set_elements(**st["sc"].element_kwargs())
        x = workloads.run_gpu(st["sc"], system=(st["pattern"], s), **_how(case))["x"]
        s.close()
        return x
    if st["path"] == "coupled":
        r = workloads.run_coupled_gpu(st["flow"], st["heat"], systems=st["systems"])
        return {"flow": r["x_flow"], "heat": r["x_heat"]}
    if st["path"] == "group":
        g, members = st["group"], st["members"]
        for s in members:
            s.copy_vector(ox.VEC_X, ox.VEC_IC)
        for k in range(case["steps"]):
            params = [workloads.step_params(sc, k, ox.DIRICHLET_SYMMETRIC) for sc in st["scs"]]
            g.step(members, params, method=ox.CG, tol=TOL, max_iter=100000)
            while g.advance() > 0:
                pass
        return [s.get_vector(ox.VEC_X) for s in members]
    ptr, col, val, b = st["dev"]
    st["x"].zero_()
    torch.cuda.current_stream().synchronize()  # the solve runs on the null stream
    ox.solve_crs_noalloc(st["n"], ptr.data_ptr(), col.data_ptr(), val.data_ptr(), b.data_ptr(),
                         st["x"].data_ptr(), tol=TOL, max_iter=100000,
                         method=ox.CG if case["method"] == "cg" else ox.BICGSTAB)
    return st["x"]


# ---- what one pass cannot do without --------------------------------------
def _work_of(case, nodes, cells, mesh, heat=False):
    """Inputs (coordinates, connectivity, coefficients, velocity, initial
    values) read once, matrix and solution written once; the element matrices'
    operations and those of a Krylov solve of about as many iterations as the
    mesh's size and process ask for."""
    elems = cells * (6 if mesh == "tet" else 1)
    npe, dim = NPE[mesh], {"line": 1, "quad": 2}.get(mesh, 3)
    nnz = ROW[mesh] * nodes
    ngp = 5 if mesh == "tet" else 3 ** dim
    cond = dim * dim if case["tensor"] else 1
    data = nodes * 8 * (dim + 2) + elems * (4 * npe + 8 * cond + 8 + (24 * ngp if heat else 0))
    iters = 60 if heat else min(5 * nodes ** (1.0 / dim), 600)
    solve = (2 if heat else 1) * iters * (2 * nnz + 12 * nodes)
    local = elems * ngp * npe * npe * (2 * dim + 2)
    return np.array([data + 8 * nnz * case["steps"], case["steps"] * (solve + local)], float)


def work(case):
    mesh, nx, ny, nz = (case[k] for k in ("mesh", "nx", "ny", "nz"))
    if case["path"] == "group":
        r = math.log(ny / nx) / max(1, case["count"] - 1)
        sides = [int(round(nx * math.exp(r * i))) for i in range(case["count"])]
        w = sum(_work_of(case, (s + 1) ** 2, s * s, mesh) for s in sides)
    elif case["path"] == "crs":
        n = nx * ny
        w = np.array([n * (5 * 12 + 4 + 24), 400 * n * (2 * 5 + 12)], float)
    else:
        shape = [s for s in (nx, ny, nz) if s]
        nodes, cells = math.prod(s + 1 for s in shape), math.prod(shape)
        w = _work_of(case, nodes, cells, mesh, case["process"] == "heat")
        if case["path"] == "coupled":
            w = w + _work_of(case, nodes, cells, mesh, True)
    return {"bytes": float(w[0]), "flops": float(w[1])}


# ---- the same solutions in plain torch, 64 bits ---------------------------
def _t(a):
    return torch.as_tensor(a, device="cuda" if torch.cuda.is_available() else "cpu")


def _unit_integrals(sc):
    """Per element type of the uniform mesh (1, or the 6 tets of a cube):
    mass [T,i,j], stiffness [T,a,b,i,j], int dN_i/dx_a [T,a,i] and
    int N_i dN_j/dx_a [T,a,i,j]."""
    m = sc.mesh
    T = 6 if m.etype == ox.TET4 else 1
    out = []
    for t in range(T):
        X = np.stack([m.x[m.conn[t]], m.y[m.conn[t]], m.z[m.conn[t]]], 1)[:, :m.dim]
        if T == 6:
            P = np.concatenate([np.ones((4, 1)), X], 1)
            g, vol = np.linalg.inv(P)[1:], abs(np.linalg.det(P)) / 6.0
            M = vol / 20.0 * (np.ones((4, 4)) + np.eye(4))
            out.append((M, vol * np.einsum("ai,bj->abij", g, g), vol * g,
                        vol / 4.0 * np.repeat(g[:, None, :], 4, 1)))
            continue
        lo, hi = X.min(0), X.max(0)
        h = hi - lo
        s = np.sign(X - (lo + hi) / 2)
        gp, gw = np.polynomial.legendre.leggauss(3)
        M = S = D = A = 0.0
        for q in np.ndindex(*[3] * m.dim):
            f = 1.0 + s * gp[list(q)]
            N = np.prod(f / 2, 1)
            g = np.stack([s[:, a] / h[a] * np.prod(np.delete(f, a, 1) / 2, 1)
                          for a in range(m.dim)])
            w = np.prod(gw[list(q)]) * np.prod(h / 2)
            M = M + w * np.outer(N, N)
            S = S + w * np.einsum("ai,bj->abij", g, g)
            D = D + w * g
            A = A + w * np.einsum("i,aj->aij", N, g)
        out.append((M, S, D, A))
    return [np.stack(v) for v in zip(*out)]


def _exact_step(sc, st, u_old, vel=None):
    """The step's solution: matrix as [n, offsets], Dirichlet values eliminated,
    Krylov iteration with restarts until the residual is rounding."""
    m = sc.mesh
    M, S, D, A = (_t(v) for v in _unit_integrals(sc))
    T, npe, dim, n = M.shape[0], m.npe, m.dim, m.n_nodes
    conn = _t(m.conn).reshape(-1, T, npe)
    K = _t(sc.cond).reshape(-1, T, sc.cond_stride) * (sc.tuf / sc.mu)
    K = K.reshape(-1, T, dim, dim) if sc.cond_stride > 1 else K[..., None] * torch.eye(dim).to(K)
    mass = (0.0 if st.steady else 1.0 / st.dt) * _t(sc.mass_coef).reshape(-1, T)
    offs, where = torch.unique(conn[0][:, None, :] - conn[0][:, :, None], return_inverse=True)
    lhs = torch.zeros(len(offs), n, dtype=torch.float64, device=M.device)
    rhs = torch.zeros(n, dtype=torch.float64, device=M.device)
    for t in range(T):
        for i in range(npe):
            for j in range(npe):
                L = (K[:, t] * S[t, :, :, i, j]).sum((1, 2))
                if vel is not None:
                    L = L + sc.adv_coef * (vel[:, t] * A[t, :, i, j]).sum(1)
                mm = mass[:, t] * M[t, i, j]
                lhs[where[t, i, j]].index_add_(0, conn[:, t, i], mm + st.theta * L)
                rhs.index_add_(0, conn[:, t, i],
                               (mm - (1.0 - st.theta) * L) * u_old[conn[:, t, j]])
            if sc.rho_g:
                rhs.index_add_(0, conn[:, t, i], -sc.rho_g * (K[:, t, :, -1] * D[t, :, i]).sum(1))
    if len(sc.st_idx):
        rhs.index_add_(0, _t(sc.st_idx), _t(sc.st_val))
    known = torch.zeros(n, dtype=torch.float64, device=M.device)
    known[_t(sc.bc_idx)] = _t(sc.bc_val)
    free = torch.ones(n, dtype=torch.float64, device=M.device)
    free[_t(sc.bc_idx)] = 0.0
    cols = (torch.arange(n, device=M.device)[:, None] + offs).clamp(0, n - 1)
    return _solve(lhs.T.contiguous(), cols, rhs, offs.tolist().index(0), known, free,
                  u_old, vel is None)


def _solve(a, cols, rhs, centre, known, free, x0, symmetric):
    def mul(v):
        return (a * v[cols]).sum(1)

    inv = free / a[:, centre]
    x = known + free * x0
    stop = 1e-30 * torch.dot(rhs, rhs)
    for _ in range(4):
        r = free * (rhs - mul(x))
        floor = 1e-28 * torch.dot(r, r) + stop
        e = torch.zeros_like(r)
        if symmetric:
            p = inv * r
            rz = torch.dot(r, p)
            for it in range(20000):
                q = free * mul(p)
                alpha = rz / torch.dot(p, q)
                e = e + alpha * p
                r = r - alpha * q
                if it % 10 == 9 and float(torch.dot(r, r)) <= float(floor):
                    break
                z = inv * r
                new = torch.dot(r, z)
                p, rz = z + (new / rz) * p, new
        else:
            r0, p, rho = r.clone(), r, torch.dot(r, r)
            for it in range(5000):
                if float(torch.dot(r, r)) <= float(floor):
                    break
                v = free * mul(inv * p)
                alpha = rho / torch.dot(r0, v)
                s = r - alpha * v
                w = free * mul(inv * s)
                ww = torch.dot(w, w)
                if float(ww) == 0.0:
                    e = e + alpha * inv * p
                    break
                om = torch.dot(w, s) / ww
                e = e + alpha * inv * p + om * inv * s
                r = s - om * w
                new = torch.dot(r0, r)
                p = r + (new / rho) * (alpha / om) * (p - om * v)
                rho = new
        x = x + e
    return x


def _exact_steps(sc):
    u = _t(sc.u0)
    vel = None
    if sc.vel is not None:  # one velocity per element: any Gauss point's
        vel = _t(np.ascontiguousarray(sc.vel[:, :, 0])).reshape(-1, 6, 3)
    for st in sc.steps:
        u = _exact_step(sc, st, u, vel)
    return u


def exact(case, seed):
    if case["path"] == "crs":
        ptr, col, val, b = _crs(case, seed)
        n, nx = b.size, case["nx"]
        row = np.repeat(np.arange(n), np.diff(ptr))
        offs = np.array([-nx, -1, 0, 1, nx])
        a = np.zeros((n, 5))
        a[row, np.searchsorted(offs, col - row)] = val
        cols = _t((np.arange(n)[:, None] + offs).clip(0, n - 1))
        one = torch.ones(n, dtype=torch.float64, device=cols.device)
        return _solve(_t(a), cols, _t(b), 2, 0 * one, one, 0 * one,
                      case["method"] == "cg").cpu()
    if case["path"] == "group":
        return [_exact_steps(sc).cpu() for sc in _group(case, seed)]
    if case["path"] == "coupled":
        flow, heat = _coupled(case, seed)
        m = flow.mesh
        grad = _unit_integrals(flow)[2]
        vol = m.h[0] * m.h[1] * m.h[2] / 6.0
        conn = _t(m.conn).reshape(-1, 6, 4)
        uf, uh = _t(flow.u0), _t(heat.u0)
        k = _t(flow.cond).reshape(-1, 6, 1) / flow.mu
        ez = _t(np.array([0.0, 0.0, flow.rho_g]))
        for sf, sh in zip(flow.steps, heat.steps):
            uf = _exact_step(flow, sf, uf)
            v = -k * (torch.einsum("eti,tai->eta", uf[conn], _t(grad) / vol) + ez)
            uh = _exact_step(heat, sh, uh, v)
        return {"flow": uf.cpu(), "heat": uh.cpu()}
    return _exact_steps(_scenario(case, seed)).cpu()
