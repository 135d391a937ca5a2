"""The work whose speed is measured: what a program that uses this package has the
GPU do, from the smallest solve to a batch of served requests.

A case is one call sequence through the public Python layer (iron_amd.fem,
iron_amd.finite_elasticity, iron_amd.serving) at one size.  The families, with the
range of sizes that the listed case stands for:

  pass       one linear solve as Problem.Solve() runs it: assembly, solver values, RHS,
             Jacobi CG in the precision fem.auto_precision picks, field update, reactions
             (generated scalar meshes, trilinear 8..64 or triquadratic 6..48 elements per
             direction, lognormal conductivity)
  cg         the Krylov layer alone: FP64 Jacobi CG on a three-component elasticity
             matrix (3x3 node blocks), boxes of up to 96x32x32 trilinear elements
  assemble   element integration into the equations CSR of a generated mesh whose nodes
             were moved: triquadratic and trilinear diffusion, trilinear elasticity
  scatter    the same through the coloured scatter, which meshes that are not generated
             grids take
  reactions  the per-solve sparse work around the Krylov solver: the lifted RHS and both
             back-substitutions (iron's stored values and the correct reactions)
  mr_step    the two element passes of a Mooney-Rivlin Newton step: residual + Jacobian at
             a state, and the line search's residual at a trial state
  mr_linear  the linear solve of a Newton step, GMRES on the FP64 matrix or MINRES on its
             FP32 values (Newton's default), 4..12 triquadratic elements per direction
  serve      a batch of independent requests of mixed size through the grouped server

Tolerances are 1e-10 (the 16^3 Laplace configuration's) where a case solves a linear
system to completion.  Coefficients, states and right-hand sides come from the seed.
"""
import math

import numpy as np
import torch

from iron_amd import basis, fem, finite_elasticity as fe, mesh, serving

DEV = "cuda:0"


def listed():
    return [
        # the smallest solve a user runs (the 16^3 Laplace configuration): launches and latency
        dict(name="pass_q1_16", op="pass", order=1, nx=16, ny=16, nz=16, rtol=1e-10),
        # the headline problem, 48^3 triquadratic diffusion, mixed precision by "auto"
        dict(name="pass_q2_48", op="pass", order=2, nx=48, ny=48, nz=48, rtol=1e-10),
        # the Krylov solve of the 96x32x32 elasticity cantilever: long, FP64, node blocks
        dict(name="cg_elastic_96", op="cg", nx=96, ny=32, nz=32, rtol=1e-10),
        # element integration at full size, every kind the structured assembly takes
        dict(name="assemble_q2_48", op="assemble", kind="scalar", order=2, nx=48, ny=48, nz=48),
        dict(name="assemble_q1_odd", op="assemble", kind="scalar", order=1, nx=61, ny=47, nz=53),
        dict(name="assemble_elastic_odd", op="assemble", kind="elastic", order=1, nx=63, ny=41, nz=38),
        # meshes that are not generated grids
        dict(name="scatter_q2_odd", op="scatter", order=2, nx=23, ny=19, nz=21),
        # RHS lifting and back-substitution on the equations CSR
        dict(name="reactions_q2_odd", op="reactions", order=2, nx=37, ny=41, nz=33),
        # the 12^3 Q2/Q1 Mooney-Rivlin configuration: element passes and both linear solvers
        dict(name="mr_step_12", op="mr_step", nx=12, ny=12, nz=12),
        dict(name="mr_gmres_12", op="mr_linear", solver="gmres", restart=256, nx=12, ny=12, nz=12, rtol=1e-8),
        dict(name="mr_minres_12", op="mr_linear", solver="minres", restart=1, nx=12, ny=12, nz=12, rtol=1e-8),
        # the served stream: boxes of 8..64 elements per direction, all waiting at the start
        dict(name="serve_16", op="serve", requests=16, lo=8, hi=64, rtol=1e-10),
    ]


def _size(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["pass", "pass", "cg", "assemble", "assemble", "scatter", "reactions", "mr_step", "mr_linear",
                     "serve"])

    def box(lo, hi):
        return dict(nx=_size(rng, lo, hi), ny=_size(rng, lo, hi), nz=_size(rng, lo, hi))

    if op == "pass":
        order = rng.choice([1, 2])
        return dict(op=op, order=order, rtol=1e-10, **(box(8, 64) if order == 1 else box(6, 48)))
    if op == "cg":
        return dict(op=op, nx=_size(rng, 8, 96), ny=_size(rng, 6, 32), nz=_size(rng, 6, 32), rtol=1e-10)
    if op == "assemble":
        kind, order = rng.choice([("scalar", 2), ("scalar", 1), ("elastic", 1)])
        return dict(op=op, kind=kind, order=order, **(box(6, 48) if order == 2 else box(8, 64)))
    if op == "scatter":
        return dict(op=op, order=2, **box(6, 28))
    if op == "reactions":
        return dict(op=op, order=2, **box(6, 42))
    if op == "mr_step":
        return dict(op=op, **box(3, 12))
    if op == "mr_linear":
        solver, restart = rng.choice([("gmres", 256), ("gmres", 100), ("minres", 1)])
        return dict(op=op, solver=solver, restart=restart, rtol=1e-8, **box(4, 10))
    return dict(op=op, requests=rng.randint(2, 16), lo=8, hi=_size(rng, 16, 48), rtol=1e-10)


# ------------------------------------------------------------------ inputs
def _ne(case):
    return case["nx"], case["ny"], case["nz"]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(n, g):
    return torch.randn(n, dtype=torch.float64, device=DEV, generator=g)


def _material(E, g):
    """Orthotropic material [E][6]: lognormal moduli, Poisson ratios about 0.3."""
    z = 10.0 * torch.exp(0.3 * _normal((E, 3), g))
    nu = 0.3 + 0.01 * torch.rand((E, 3), dtype=torch.float64, device=DEV, generator=g)
    return torch.cat([z, nu], dim=1).contiguous()


def _isotropic(E, g):
    z = 10.0 * torch.exp(0.3 * _normal(E, g))
    nu = torch.full_like(z, 0.3)
    return torch.stack([z, z, z, nu, nu, nu], dim=1).contiguous()


def _moved(X, ne, order, seed):
    """Node coordinates with every node moved by up to 0.1 of the node spacing."""
    h = 1.0 / (order * np.array(ne, dtype=np.float64))
    return np.ascontiguousarray(X + (np.random.default_rng(seed).random(X.shape) * 0.2 - 0.1) * h)


def _faces(X):
    return np.any((X < 1e-12) | (np.abs(X - 1.0) < 1e-12), axis=1)


def _ends(X):
    return (X[:, 0] < 1e-12) | (np.abs(X[:, 0] - 1.0) < 1e-12)


def _scalar_setup(case, coords=None, grid=True):
    ne, order = _ne(case), case["order"]
    b = basis.basis(3, order)
    m = mesh.RegularMesh(ne, [b], (1.0, 1.0, 1.0))
    dm = mesh.DofMap(m, [0])
    csr = fem.CSRStructure(dm.element_dofs(), dm.num_dofs, DEV, colours=mesh.structured_colours(m))
    X = m.coords if coords is None else coords(m.coords)
    return m, X, csr, fem.ScalarAssembler(b, X, m.elem_nodes[0], csr, grid=ne if grid else None)


def _prepare_pass(case, seed):
    g = _gen(seed)
    m, X, csr, asm = _scalar_setup(case)
    E = m.num_elements
    # trilinear: u = 0 and 1 on the two x faces; triquadratic: source 1, u = 0 on every face
    q1 = case["order"] == 1
    fixed = _ends(X) if q1 else _faces(X)
    u0 = torch.as_tensor(np.where(fixed & (X[:, 0] > 0.5), 1.0, 0.0) if q1 else np.zeros(csr.n), device=DEV)
    red = fem.DirichletReduction(csr, fixed)
    S = fem.SolverMatrix(red)
    return dict(csr=csr, asm=asm, red=red, S=S, ws=fem.KrylovWorkspace(red.n_free, DEV), rtol=case["rtol"],
                mixed=fem.auto_precision(1, S.stored) == "mixed", kappa=_normal(E, g).exp(),
                source=None if q1 else torch.ones(E, dtype=torch.float64, device=DEV), u0=u0, v=csr.zeros(fem.F64),
                src=None if q1 else torch.zeros(csr.n, dtype=torch.float64, device=DEV), u=torch.empty_like(u0),
                s64=torch.empty(max(S.stored, 1), dtype=torch.float64, device=DEV),
                s32=torch.empty(max(S.stored, 1), dtype=torch.float32, device=DEV),
                b=torch.empty(red.n_free, dtype=torch.float64, device=DEV),
                x=torch.zeros(red.n_free, dtype=torch.float64, device=DEV), R=torch.empty_like(u0))


def _run_pass(P):
    v, S, red, x = P["v"], P["S"], P["red"], P["x"]
    P["asm"].assemble(v, kappa=P["kappa"], source=P["source"], src_vec=P["src"])
    if P["mixed"]:
        S.gather2(v, out64=P["s64"], out32=P["s32"])
    else:
        S.gather(v, fem.F64, out=P["s64"])
    P["u"].copy_(P["u0"])
    red.rhs(v, P["u"], src=P["src"], out=P["b"])
    x.zero_()
    if P["mixed"]:
        fem.refine(S, P["s64"], P["s32"], P["b"], x, P["rtol"], 200000, P["ws"])
    else:
        fem.cg(S, P["s64"], P["b"], x, P["rtol"], 200000, P["ws"])
    red.field_update(x, P["u"])
    fem.backsubstitute(P["csr"], v, P["u"], src=P["src"], out=P["R"])
    return dict(u=P["u"], R=P["R"])


def _traction(ne):
    """Nodal forces [3 N] of t_z = -1 on the x end face of an x-fastest node grid."""
    Nx, Ny, Nz = (n + 1 for n in ne)
    cy, cz = np.ones(Ny), np.ones(Nz)
    cy[[0, -1]] = cz[[0, -1]] = 0.5
    f = np.zeros((3, Nz, Ny, Nx))
    f[2, :, :, -1] = -np.outer(cz, cy) / (ne[1] * ne[2])
    return f.reshape(-1)


def _prepare_cg(case, seed):
    g = _gen(seed)
    ne = _ne(case)
    b = basis.basis(3, 1)
    m = mesh.RegularMesh(ne, [b], (3.0, 1.0, 1.0))
    dm = mesh.DofMap(m, [0, 0, 0])
    csr = fem.CSRStructure(dm.element_dofs(), dm.num_dofs, DEV, colours=mesh.structured_colours(m))
    asm = fem.ElasticAssembler(b, m.coords, m.elem_nodes[0], csr, grid=ne)
    red = fem.DirichletReduction(csr, np.tile(m.coords[:, 0] == 0.0, 3))
    S = fem.SolverMatrix(red, interleave=(3, m.num_nodes(0)), block=True)
    v = asm.assemble(csr.zeros(fem.F64), _isotropic(m.num_elements, g))
    f = torch.as_tensor(_traction(ne), device=DEV)
    bvec = red.rhs(v, torch.zeros(csr.n, dtype=torch.float64, device=DEV), rhs=f)
    return dict(S=S, vals=S.gather(v), b=bvec, ws=fem.KrylovWorkspace(red.n_free, DEV), rtol=case["rtol"],
                x=torch.zeros_like(bvec))


def _run_cg(P):
    P["x"].zero_()
    fem.cg(P["S"], P["vals"], P["b"], P["x"], P["rtol"], 200000, P["ws"])
    return P["x"]


def _prepare_assemble(case, seed):
    g = _gen(seed)
    ne, order = _ne(case), case["order"]
    grid = case["op"] == "assemble"
    moved = lambda X: _moved(X, ne, order, seed)  # noqa: E731
    if case.get("kind") == "elastic":
        b = basis.basis(3, 1)
        m = mesh.RegularMesh(ne, [b], (1.0, 1.0, 1.0))
        dm = mesh.DofMap(m, [0, 0, 0])
        csr = fem.CSRStructure(dm.element_dofs(), dm.num_dofs, DEV, colours=mesh.structured_colours(m))
        asm = fem.ElasticAssembler(b, moved(m.coords), m.elem_nodes[0], csr, grid=ne)
        return dict(asm=asm, v=csr.zeros(fem.F64), material=_material(m.num_elements, g))
    m, _, csr, asm = _scalar_setup(case, moved, grid)
    E = m.num_elements
    return dict(asm=asm, v=csr.zeros(fem.F64), material=None, grid=grid, kappa=_normal(E, g).exp(),
                source=_normal(E, g), src=torch.zeros(csr.n, dtype=torch.float64, device=DEV))


def _run_assemble(P):
    if P["material"] is not None:
        return P["asm"].assemble(P["v"], P["material"])
    if not P["grid"]:  # the coloured scatter adds into its outputs, the structured assembly writes them
        P["v"].zero_()
        P["src"].zero_()
    P["asm"].assemble(P["v"], kappa=P["kappa"], source=P["source"], src_vec=P["src"])
    return dict(v=P["v"], src=P["src"])


def _prepare_reactions(case, seed):
    g = _gen(seed)
    m, X, csr, asm = _scalar_setup(case)
    E = m.num_elements
    v, src = csr.zeros(fem.F64), torch.zeros(csr.n, dtype=torch.float64, device=DEV)
    asm.assemble(v, kappa=_normal(E, g).exp(), source=_normal(E, g), src_vec=src)
    red = fem.DirichletReduction(csr, _faces(X))
    return dict(csr=csr, red=red, v=v, src=src, u=_normal(csr.n, g))


def _run_reactions(P):
    csr, v, u, src = P["csr"], P["v"], P["u"], P["src"]
    return dict(b=P["red"].rhs(v, u, src=src), R_iron=fem.backsubstitute(csr, v, u, src=src, iron_compat=True),
                R=fem.backsubstitute(csr, v, u, src=src))


def _mr_state(nodes, npd, ne, g):
    """A stretched state with every deformed coordinate moved a little, and pressures."""
    X = torch.as_tensor(nodes, device=DEV)
    z = X * torch.tensor([1.1, 1.1 ** -0.5, 1.1 ** -0.5], dtype=torch.float64, device=DEV)
    h = 0.5 / torch.tensor(ne, dtype=torch.float64, device=DEV)
    z = z + 0.02 * h * _normal(tuple(X.shape), g)
    return torch.cat([z.t().reshape(-1), _normal(npd, g)]).contiguous()


def _mr_moduli(E, g):
    """c1 in [1, 3), c2 in [4, 8) per element."""
    r = torch.rand((E, 2), dtype=torch.float64, device=DEV, generator=g)
    return torch.stack([1.0 + 2.0 * r[:, 0], 4.0 + 4.0 * r[:, 1]], dim=1).contiguous()


def _mr_system(case):
    return fe.MRSystem(mesh.RegularMesh(_ne(case), [basis.basis(3, 2, 3), basis.basis(3, 1, 3)], (1.0, 1.0, 1.0)), 1,
                       fe.DEVIATORIC)


def _prepare_mr_step(case, seed):
    g = _gen(seed)
    sysm = _mr_system(case)
    material = _mr_moduli(sysm.rm.num_elements, g)
    x = _mr_state(sysm.X, sysm.npd, _ne(case), g)
    trial = x + 1e-3 * _normal(x.shape[0], g) / max(_ne(case))
    return dict(sys=sysm, material=material, x=x, trial=trial, R=torch.zeros_like(x), Rt=torch.zeros_like(x),
                J=sysm.csr.zeros())


def _run_mr_step(P):
    for k in ("R", "J", "Rt"):
        P[k].zero_()
    P["sys"].assemble(P["x"], P["material"], residual=P["R"], jac=P["J"])
    P["sys"].assemble(P["trial"], P["material"], residual=P["Rt"])
    return dict(R=P["R"], J=P["J"], Rt=P["Rt"])


def _mr_fixed(X, ndofs):
    """Rollers on x = 0, y = 0, z = 0 and the x = 1 face held in x."""
    nu = len(X)
    fixed = np.zeros(ndofs, dtype=bool)
    for c in range(3):
        fixed[c * nu:(c + 1) * nu] = X[:, c] == 0.0
    fixed[:nu] |= X[:, 0] == 1.0
    return fixed


def _prepare_mr_linear(case, seed):
    g = _gen(seed)
    sysm = _mr_system(case)
    material = _mr_moduli(sysm.rm.num_elements, g)
    x = _mr_state(sysm.X, sysm.npd, _ne(case), g)
    newton = fe.MRNewton(sysm, _mr_fixed(sysm.X, sysm.ndofs), material.cpu().numpy(), restart=case["restart"])
    R, J = torch.zeros_like(x), sysm.csr.zeros()
    sysm.assemble(x, newton.material, residual=R, jac=J)
    gm = case["solver"] == "gmres"
    b = -R.index_select(0, newton.free)
    return dict(newton=newton, gmres=gm, vals=newton.S.gather(J, fem.F64 if gm else fem.F32), b=b,
                dx=torch.zeros_like(b), rtol=case["rtol"], restart=case["restart"])


def _run_mr_linear(P):
    n, dx = P["newton"], P["dx"]
    dx.zero_()
    if P["gmres"]:
        fem.gmres(n.S, P["vals"], P["b"], dx, P["rtol"], 100000, n.ws, restart=P["restart"], pc_inv=n.pc_neg)
    else:
        fem.minres(n.S, P["vals"], P["b"], dx, P["rtol"], 100000, n.ws, pc_inv=n.pc_pos)
    return dx


def _requests(case, seed):
    """The batch: shapes are the case's (one per position), coefficients the seed's."""
    rng = np.random.default_rng(2024)
    out = []
    for i in range(case["requests"]):
        kind = "diffusion" if i % 3 else "elasticity"
        ne = tuple(int(v) for v in rng.integers(case["lo"], case["hi"] + 1, size=3))
        out.append((kind, ne, int(seed) * 1000 + i))
    return out


def _prepare_serve(case, seed):
    srv = serving.Server(hbm_budget=8e9, max_segments=64)
    return dict(srv=srv, batch=_requests(case, seed), rtol=case["rtol"])


def _run_serve(P):
    reqs = [serving.Request(i, kind, ne, s, rtol=P["rtol"]) for i, (kind, ne, s) in enumerate(P["batch"])]
    return [r.u for r in P["srv"].run(reqs)]


_FAMILIES = {"pass": (_prepare_pass, _run_pass), "cg": (_prepare_cg, _run_cg),
             "assemble": (_prepare_assemble, _run_assemble), "scatter": (_prepare_assemble, _run_assemble),
             "reactions": (_prepare_reactions, _run_reactions), "mr_step": (_prepare_mr_step, _run_mr_step),
             "mr_linear": (_prepare_mr_linear, _run_mr_linear), "serve": (_prepare_serve, _run_serve)}


def prepare(case, seed):
    prep, run_one = _FAMILIES[case["op"]]
    return run_one, prep(case, seed)


def run(state):
    return state[0](state[1])


# ------------------------------------------------------------------ work
def _pairs(n, order):
    """Node pairs that share an element along one direction of n elements."""
    return 9 * n - (n - 1) if order == 2 else 4 * n - (n - 1)


def _shape(ne, order, comps=1):
    """(elements, nodes, stored entries of the equations CSR) of a generated grid."""
    E = ne[0] * ne[1] * ne[2]
    N = math.prod(order * n + 1 for n in ne)
    return E, N, comps * comps * math.prod(_pairs(n, order) for n in ne)


# element flops: 3x3x3 / 2x2x2 Gauss integration of K = B^T W B with its geometry
_FLOPS = {("scalar", 2): 144342, ("scalar", 1): 5000, ("elastic", 1): 71424}


def _krylov_work(rows, nnz, value_bytes, vectors, iterations):
    """Every iteration reads the values once and touches its vectors once."""
    return dict(bytes=iterations * (value_bytes * nnz + value_bytes * vectors * rows), flops=iterations * 2.0 * nnz)


def work(case):
    """Bytes and flops of one pass.  The iteration counts of Jacobi CG, GMRES and MINRES are taken
    as proportional to the nodes along the longest direction, as measured on the listed cases."""
    op = case["op"]
    if op == "serve":
        total = dict(bytes=0.0, flops=0.0)
        for kind, ne, _ in _requests(case, 0):
            comps = 1 if kind == "diffusion" else 3
            _, N, nnz = _shape(ne, 1, comps)
            its = (6 if comps == 1 else 18) * (max(ne) + 1)
            for k, v in _krylov_work(comps * N, nnz, 8, 8, its).items():
                total[k] += v
        return total
    ne = _ne(case)
    order = case.get("order", 1)
    if op == "cg":
        _, N, nnz = _shape(ne, 1, 3)
        return _krylov_work(3 * N, nnz, 8, 8, 15 * (max(ne) + 1))
    if op == "mr_linear":
        _, Nu, nnz_u = _shape(ne, 2, 3)
        Np = math.prod(n + 1 for n in ne)
        its = 60 * max(ne)
        nnz = nnz_u + 2 * 3 * 27 * Np * 4
        w = _krylov_work(3 * Nu + Np, nnz, 8 if case["solver"] == "gmres" else 4, 8, its)
        if case["solver"] == "gmres":
            w["bytes"] += its * 8.0 * (3 * Nu + Np) * case["restart"] / 2
            w["flops"] += its * 4.0 * (3 * Nu + Np) * case["restart"] / 2
        return w
    if op == "mr_step":
        E, Nu, nnz_u = _shape(ne, 2, 3)
        Np = math.prod(n + 1 for n in ne)
        nnz = nnz_u + 2 * 3 * 27 * Np * 4
        return dict(bytes=8.0 * (nnz + 4 * (3 * Nu + Np)) + 4.0 * 89 * E, flops=E * (2002968.0 + 160000.0))
    E, N, nnz = _shape(ne, order, 3 if case.get("kind") == "elastic" else 1)
    asm = dict(bytes=8.0 * nnz + 24.0 * N + 4.0 * (order + 1) ** 3 * E,
               flops=float(E) * _FLOPS[(case.get("kind", "scalar"), order)])
    if op in ("assemble", "scatter"):
        return asm
    if op == "reactions":
        return dict(bytes=12.0 * nnz + 48.0 * N, flops=4.0 * nnz)
    mixed = nnz >= 16_000_000
    its = (5 if order == 2 else 3) * (order * max(ne) + 1)
    w = _krylov_work(N, nnz, 4 if mixed else 8, 8, its)
    return dict(bytes=w["bytes"] + asm["bytes"] + 20.0 * nnz, flops=w["flops"] + asm["flops"] + 4.0 * nnz)


# ------------------------------------------------------------------ exact
# The same outputs from plain torch in 64 bits: tensor-product shape functions, Gauss
# integration, sorted CSR, Krylov solves to round-off.
def _tables(order, gauss, nodes=None):
    """Shape functions N [g][a], reference gradients dN [g][a][3], weights [g] on [0,1]^3
    (first direction fastest); ``gauss`` points per direction."""
    t, w = np.polynomial.legendre.leggauss(gauss)
    t, w = 0.5 * (t + 1.0), 0.5 * w
    pts = np.linspace(0.0, 1.0, order + 1)
    V = np.linalg.inv(np.vander(pts, increasing=True))  # monomial coefficients of each function, by column
    phi = np.vander(t, order + 1, increasing=True) @ V
    d = np.zeros((len(t), order + 1))
    d[:, 1:] = np.vander(t, order, increasing=True) * np.arange(1, order + 1)
    dphi = d @ V

    def tensor(a, b, c):
        return np.einsum("zc,yb,xa->zyxcba", c, b, a).reshape(len(t) ** 3, (order + 1) ** 3)

    N = tensor(phi, phi, phi)
    dN = np.stack([tensor(dphi, phi, phi), tensor(phi, dphi, phi), tensor(phi, phi, dphi)], axis=2)
    W = np.einsum("z,y,x->zyx", w, w, w).reshape(-1)
    return tuple(torch.as_tensor(np.ascontiguousarray(v), device=DEV) for v in (N, dN, W))


def _grid(ne, order, extent=(1.0, 1.0, 1.0)):
    """Node coordinates [N][3] and element nodes [E][(order+1)^3] of a box, x fastest."""
    n = [order * k + 1 for k in ne]
    ax = [np.arange(n[k], dtype=np.float64) * (extent[k] / (n[k] - 1)) for k in range(3)]
    Z, Y, X = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    coords = np.stack([X.reshape(-1), Y.reshape(-1), Z.reshape(-1)], axis=1)
    first = (np.arange(ne[0]) * order + n[0] * (np.arange(ne[1])[:, None] * order
                                                + n[1] * np.arange(ne[2])[:, None, None] * order)).reshape(-1)
    a = np.arange(order + 1)
    local = (a + n[0] * (a[:, None] + n[1] * a[:, None, None])).reshape(-1)
    return coords, torch.as_tensor(first[:, None] + local[None, :], device=DEV)


def _geometry(X, en, dN, W):
    """dxi_j/dx_i [E][g][j][i] and |J| w [E][g]."""
    J = torch.einsum("eai,gaj->egij", X[en], dN)
    return torch.linalg.inv(J), torch.linalg.det(J).abs() * W


def _chunks(E, step=16384):
    return [slice(i, min(i + step, E)) for i in range(0, E, step)]


def _scalar_elements(X, en, order, kappa, source):
    N, dN, W = _tables(order, order + 1)
    Ke, fe_ = [], []
    for c in _chunks(len(en)):
        ji, wj = _geometry(X, en[c], dN, W)
        B = torch.einsum("gaj,egji->egia", dN, ji).reshape(wj.shape[0], -1, dN.shape[1])
        D = (wj * kappa[c, None]).repeat_interleave(3, dim=1)
        Ke.append(torch.bmm((B * D[:, :, None]).transpose(1, 2).contiguous(), B.contiguous()))
        if source is not None:
            fe_.append((wj @ N) * source[c, None])
    return torch.cat(Ke), (torch.cat(fe_) if source is not None else None)


def _elastic_elements(X, en, mat):
    """Orthotropic stiffness [E][24][24], the gradients with iron's DXI_DX index order."""
    _, dN, W = _tables(1, 2)
    out = []
    for c in _chunks(len(en)):
        ji, wj = _geometry(X, en[c], dN, W)
        B = torch.einsum("gan,egmn->egam", dN, ji)
        E1, E2, E3, v13, v23, v12 = mat[c].unbind(1)
        gam = 1.0 / (1.0 - v12 * v12 - v23 * v23 - v13 * v13 - 2.0 * v12 * v23 * v13)
        C = torch.zeros((len(E1), 3, 3, 3, 3), dtype=torch.float64, device=DEV)
        nrm = [[E1 * (1 - v23 * v23) * gam, E1 * (v12 + v13 * v23) * gam, E1 * (v13 + v12 * v23) * gam],
               [None, E2 * (1 - v13 * v13) * gam, E2 * (v23 + v12 * v13) * gam], [None, None, E3 * (1 - v12 * v12) * gam]]
        shear = {(0, 1): E3 / (2 * (1 + v12)), (0, 2): E2 / (2 * (1 + v23)), (1, 2): E1 / (2 * (1 + v13))}
        for i in range(3):
            C[:, i, i, i, i] = nrm[i][i]
            for j in range(i + 1, 3):
                C[:, i, i, j, j] = C[:, j, j, i, i] = nrm[i][j]
                s = shear[(i, j)]
                C[:, i, j, i, j] = C[:, j, i, j, i] = C[:, i, j, j, i] = C[:, j, i, i, j] = s
        # K[(i,a)][(j,b)] = sum w B[a][k] C[i][k][j][l] B[b][l]
        U = torch.einsum("egak,eikjl,eg->eiajgl", B, C, wj)
        out.append(torch.einsum("eiajgl,egbl->eiajb", U, B).reshape(len(E1), 24, 24))
    return torch.cat(out)


class _Csr:
    """Sorted CSR of element matrices."""

    def __init__(self, ed, Ke, n):
        key = ((ed[:, :, None] * n) + ed[:, None, :]).reshape(-1)
        uniq, inv = torch.unique(key, return_inverse=True)
        self.n = n
        self.vals = torch.zeros(len(uniq), dtype=torch.float64, device=DEV).index_add_(0, inv, Ke.reshape(-1))
        self.row, self.col = uniq // n, uniq % n
        self.ptr = torch.searchsorted(self.row, torch.arange(n + 1, device=DEV))

    def free(self, free):
        """The free x free part as a torch CSR tensor."""
        rank = torch.full((self.n,), -1, dtype=torch.int64, device=DEV)
        rank[free] = torch.arange(len(free), device=DEV)
        r, c = rank[self.row], rank[self.col]
        k = (r >= 0) & (c >= 0)
        m = len(free)
        ptr = torch.searchsorted(r[k], torch.arange(m + 1, device=DEV))
        return torch.sparse_csr_tensor(ptr, c[k], self.vals[k], (m, m))

    def times(self, u, col=None):
        return torch.zeros(self.n, dtype=torch.float64, device=DEV).index_add_(
            0, self.row, self.vals * u[self.col if col is None else col])


def _vector(ed, f, n):
    return torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, ed.reshape(-1), f.reshape(-1))


def _solve_spd(A, diag, b, tol=1e-14):
    """Jacobi CG, restarted from the true residual until it stops falling."""
    x = torch.zeros_like(b)
    bn, last = float(b.norm()), math.inf
    for _ in range(4):
        r = b - A @ x
        rn = float(r.norm())
        if rn <= tol * bn or rn > 0.3 * last:
            break
        last = rn
        z = r / diag
        p, rz = z.clone(), torch.dot(r, z)
        for it in range(20000):
            q = A @ p
            a = rz / torch.dot(p, q)
            x += a * p
            r -= a * q
            z = r / diag
            new = torch.dot(r, z)
            p = z + (new / rz) * p
            rz = new
            if it % 50 == 49 and float(r.norm()) <= 0.3 * tol * bn:
                break
    return x


def _solve_symmetric(A, diag, b, tol=1e-14):
    """Preconditioned MINRES (Paige and Saunders 1975) on the true residual, again and again
    until it stops falling."""
    x = torch.zeros_like(b)
    bn, last = float(b.norm()), math.inf
    for _ in range(6):
        r = b - A @ x
        rn = float(r.norm())
        if rn <= tol * bn or rn > 0.3 * last:
            break
        last = rn
        x = x + _minres(A, diag, r, 1e-7)
    return x


def _minres(A, diag, b, tol):
    x, w, w2 = torch.zeros_like(b), torch.zeros_like(b), torch.zeros_like(b)
    r1 = r2 = b
    y = b / diag
    beta1 = beta = float(torch.dot(b, y)) ** 0.5
    oldb, dbar, eps, phibar, cs, sn = 0.0, 0.0, 0.0, beta1, -1.0, 0.0
    for it in range(20000):
        v = y / beta
        y = A @ v
        if it:
            y = y - (beta / oldb) * r1
        alfa = float(torch.dot(v, y))
        y = y - (alfa / beta) * r2
        r1, r2 = r2, y
        y = r2 / diag
        oldb, beta = beta, float(torch.dot(r2, y)) ** 0.5
        olde, delta, gbar = eps, cs * dbar + sn * alfa, sn * dbar - cs * alfa
        eps, dbar = sn * beta, -cs * beta
        gamma = math.hypot(gbar, beta)
        cs, sn = gbar / gamma, beta / gamma
        phi, phibar = cs * phibar, sn * phibar
        w1, w2 = w2, w
        w = (v - olde * w1 - delta * w2) / gamma
        x = x + phi * w
        if phibar <= tol * beta1:
            break
    return x


def _solve_reduced(M, fixed, u0, f):
    """u with the fixed DOFs at u0 and the free rows of M u = f solved."""
    free = torch.nonzero(~fixed).reshape(-1)
    b = (f - M.times(torch.where(fixed, u0, 0.0)))[free]
    A = M.free(free)
    d = torch.zeros(M.n, dtype=torch.float64, device=DEV)
    on = M.row == M.col
    d[M.row[on]] = M.vals[on]
    u = torch.where(fixed, u0, 0.0)
    u[free] = _solve_spd(A, d[free], b)
    return u


def _exact_pass(case, seed):
    g = _gen(seed)
    ne, order = _ne(case), case["order"]
    Xh, en = _grid(ne, order)
    E, n = len(en), len(Xh)
    kappa = _normal(E, g).exp()
    X = torch.as_tensor(Xh, device=DEV)
    q1 = order == 1
    Ke, fv = _scalar_elements(X, en, order, kappa, None if q1 else torch.ones(E, dtype=torch.float64, device=DEV))
    f = torch.zeros(n, dtype=torch.float64, device=DEV) if q1 else _vector(en, fv, n)
    M = _Csr(en, Ke, n)
    del Ke
    fixed = torch.as_tensor(_ends(Xh) if q1 else _faces(Xh), device=DEV)
    u0 = torch.where(fixed & (X[:, 0] > 0.5), 1.0, 0.0).double() if q1 else torch.zeros(n, dtype=torch.float64, device=DEV)
    u = _solve_reduced(M, fixed, u0, f)
    return dict(u=u, R=M.times(u) - f)


def _elastic_solution(ne, mat):
    Xh, en = _grid(ne, 1, (3.0, 1.0, 1.0))
    N = len(Xh)
    Ke = _elastic_elements(torch.as_tensor(Xh, device=DEV), en, mat)
    M = _Csr(torch.cat([en, en + N, en + 2 * N], dim=1), Ke, 3 * N)
    fixed = torch.as_tensor(np.tile(Xh[:, 0] == 0.0, 3), device=DEV)
    zero = torch.zeros(3 * N, dtype=torch.float64, device=DEV)
    return fixed, _solve_reduced(M, fixed, zero, torch.as_tensor(_traction(ne), device=DEV))


def _exact_cg(case, seed):
    ne = _ne(case)
    fixed, u = _elastic_solution(ne, _isotropic(ne[0] * ne[1] * ne[2], _gen(seed)))
    return u[~fixed]


def _exact_assemble(case, seed):
    g = _gen(seed)
    ne, order = _ne(case), case["order"]
    Xh, en = _grid(ne, order)
    E, N = len(en), len(Xh)
    X = torch.as_tensor(_moved(Xh, ne, order, seed), device=DEV)
    if case.get("kind") == "elastic":
        Ke = _elastic_elements(X, en, _material(E, g))
        return _Csr(torch.cat([en, en + N, en + 2 * N], dim=1), Ke, 3 * N).vals
    kappa, source = _normal(E, g).exp(), _normal(E, g)
    Ke, fv = _scalar_elements(X, en, order, kappa, source)
    return dict(v=_Csr(en, Ke, N).vals, src=_vector(en, fv, N))


def _exact_reactions(case, seed):
    g = _gen(seed)
    ne, order = _ne(case), case["order"]
    Xh, en = _grid(ne, order)
    E, N = len(en), len(Xh)
    Ke, fv = _scalar_elements(torch.as_tensor(Xh, device=DEV), en, order, _normal(E, g).exp(), _normal(E, g))
    M, f = _Csr(en, Ke, N), _vector(en, fv, N)
    u = _normal(N, g)
    fixed = torch.as_tensor(_faces(Xh), device=DEV)
    inrow = torch.arange(len(M.vals), device=DEV) - M.ptr[M.row]
    return dict(b=(f - M.times(torch.where(fixed, u, 0.0)))[~fixed], R_iron=M.times(u, inrow) - f, R=M.times(u) - f)


def _mr_elements(ne, X, en, x, c, jac):
    """Residual [E][89] and Jacobian [E][89][89] of W = c1 (I1bar - 3) + c2 (I2bar - 3) + p (J - 1)."""
    nu = len(X)
    _, dN, W = _tables(2, 3)
    # trilinear pressure functions at the 3x3x3 points
    Np = _tables(1, 3)[0]
    corner = [i + 3 * (j + 3 * k) for k in (0, 2) for j in (0, 2) for i in (0, 2)]
    pn = torch.unique(en[:, corner])
    ep = torch.searchsorted(pn, en[:, corner])
    ed = torch.cat([en, en + nu, en + 2 * nu, ep + 3 * nu], dim=1)
    E = len(en)
    ji, wj = _geometry(X, en, dN, W)
    GX = torch.einsum("gam,egmK->egaK", dN, ji)
    z = torch.stack([x[en + k * nu] for k in range(3)], dim=2)  # [E][a][i]
    F = torch.einsum("eai,egaK->egiK", z, GX).detach().requires_grad_(True)
    p = torch.einsum("gq,eq->eg", Np, x[ep + 3 * nu])
    Jd = torch.linalg.det(F)
    C = torch.einsum("egki,egkj->egij", F, F)
    I1 = C.diagonal(dim1=2, dim2=3).sum(-1)
    I2 = 0.5 * (I1 * I1 - (C * C).sum((2, 3)))
    Wd = c[:, :1] * Jd ** (-2.0 / 3.0) * I1 + c[:, 1:] * Jd ** (-4.0 / 3.0) * I2 + p * Jd
    P = torch.autograd.grad(Wd.sum(), F, create_graph=True)[0]
    JG = torch.autograd.grad(torch.linalg.det(F).sum(), F)[0]
    Ru = torch.einsum("eg,egaK,egiK->eia", wj, GX, P.detach()).reshape(E, 81)
    Rp = torch.einsum("eg,eg,gq->eq", wj, Jd.detach() - 1.0, Np)
    R = torch.cat([Ru, Rp], dim=1)
    if not jac:
        return ed, R, None
    K = torch.zeros((E, 89, 89), dtype=torch.float64, device=DEV)
    for i in range(3):
        U = torch.zeros((E, 27, 27, 3, 3), dtype=torch.float64, device=DEV)  # [e][g][a][j][L]
        for k in range(3):
            A = torch.autograd.grad(P[:, :, i, k].sum(), F, retain_graph=True)[0]
            U += GX[:, :, :, k, None, None] * (wj[:, :, None, None] * A)[:, :, None]
        for j in range(3):
            K[:, 27 * i:27 * i + 27, 27 * j:27 * j + 27] = torch.einsum("egaL,egbL->eab", U[:, :, :, j], GX)
        up = torch.einsum("eg,egaK,egK,gq->eaq", wj, GX, JG[:, :, i], Np)
        K[:, 27 * i:27 * i + 27, 81:] = up
        K[:, 81:, 27 * i:27 * i + 27] = up.transpose(1, 2)
    return ed, R, K


def _mr_inputs(case, seed):
    g = _gen(seed)
    ne = _ne(case)
    Xh, en = _grid(ne, 2)
    npd = math.prod(n + 1 for n in ne)
    c = _mr_moduli(len(en), g)
    x = _mr_state(Xh, npd, ne, g)
    return g, ne, Xh, en, c, x


def _exact_mr_step(case, seed):
    g, ne, Xh, en, c, x = _mr_inputs(case, seed)
    X = torch.as_tensor(Xh, device=DEV)
    trial = x + 1e-3 * _normal(x.shape[0], g) / max(ne)
    ed, R, K = _mr_elements(ne, X, en, x, c, True)
    _, Rt, _ = _mr_elements(ne, X, en, trial, c, False)
    n = x.shape[0]
    return dict(R=_vector(ed, R, n), J=_Csr(ed, K, n).vals, Rt=_vector(ed, Rt, n))


def _exact_mr_linear(case, seed):
    _, ne, Xh, en, c, x = _mr_inputs(case, seed)
    ed, R, K = _mr_elements(ne, torch.as_tensor(Xh, device=DEV), en, x, c, True)
    n = x.shape[0]
    M, r = _Csr(ed, K, n), _vector(ed, R, n)
    free = torch.nonzero(torch.as_tensor(~_mr_fixed(Xh, n), device=DEV)).reshape(-1)
    A = M.free(free)
    # diagonal preconditioner: |a_ii|, and on the zero pressure diagonal the sums k_qj^2 / |a_jj|
    d = torch.zeros(n, dtype=torch.float64, device=DEV)
    on = M.row == M.col
    d[M.row[on]] = M.vals[on].abs()
    up = (M.row >= n - math.prod(k + 1 for k in ne)) & (d[M.col] > 0)
    d.index_add_(0, M.row[up], M.vals[up] ** 2 / d[M.col[up]])
    return _solve_symmetric(A, d[free], -r[free])


def _exact_serve(case, seed):
    out = []
    for kind, ne, s in _requests(case, seed):
        E = ne[0] * ne[1] * ne[2]
        z = torch.randn(E, dtype=torch.float64, generator=_gen(s), device=DEV).exp_()
        if kind == "diffusion":
            Xh, en = _grid(ne, 1)
            X = torch.as_tensor(Xh, device=DEV)
            M = _Csr(en, _scalar_elements(X, en, 1, z, None)[0], len(Xh))
            fixed = torch.as_tensor(_ends(Xh), device=DEV)
            u0 = torch.where(fixed & (X[:, 0] > 0.5), 1.0, 0.0).double()
            out.append(_solve_reduced(M, fixed, u0, torch.zeros_like(u0)))
        else:
            nu = torch.full_like(z, 0.3)
            out.append(_elastic_solution(ne, torch.stack([10 * z, 10 * z, 10 * z, nu, nu, nu], dim=1))[1])
    return out


_EXACT = {"pass": _exact_pass, "cg": _exact_cg, "assemble": _exact_assemble, "scatter": _exact_assemble,
          "reactions": _exact_reactions, "mr_step": _exact_mr_step, "mr_linear": _exact_mr_linear,
          "serve": _exact_serve}


def exact(case, seed):
    return _EXACT[case["op"]](case, seed)
