"""GMRES whose Hessenberg columns are rotated within the next iteration's dot products:
restart lengths around the chunk of eight iterations after which the column is rotated
by a launch of its own, around the eight rotations applied at a time, and with the second
Gram-Schmidt pass, against a dense solve; and MINRES beside them."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _system(ne=(7, 5, 4)):
    from iron_amd import basis, fem, mesh
    b = basis.basis(3, 1, 2)
    m = mesh.RegularMesh(ne, [b], (1.0, 1.0, 1.0))
    dm = mesh.DofMap(m, [0])
    X = m.coords
    fixed = (X[:, 0] == 0.0) | (X[:, 0] == 1.0)
    csr = fem.CSRStructure(dm.element_dofs(), dm.num_dofs)
    kappa = np.exp(0.5 * np.random.default_rng(2).standard_normal(m.num_elements))
    v = csr.zeros()
    fem.ScalarAssembler(b, X, m.elem_nodes[0], csr).assemble(v, kappa=torch.as_tensor(kappa, device="cuda"))
    red = fem.DirichletReduction(csr, fixed)
    u = torch.as_tensor(np.where(X[:, 0] == 1.0, 1.0, 0.0), device="cuda")
    rhs = red.rhs(v, u)
    rp, col = red.row_ptr.cpu().long(), red.col[:red.nnz].cpu().long()
    rows = torch.repeat_interleave(torch.arange(red.n_free), rp[1:] - rp[:-1])
    A = torch.zeros(red.n_free, red.n_free, dtype=torch.float64)
    A[rows, col] = fem.SolverMatrix(red, "csr").gather(v)[:red.nnz].cpu()
    return fem, red, v, rhs, torch.linalg.solve(A, rhs.cpu())


@pytest.mark.parametrize("refine", [0, 1])
@pytest.mark.parametrize("restart", [2, 7, 8, 9, 16, 17, 18, 33, 256])
def test_gmres_restart_lengths(restart, refine):
    from iron_amd import _lib
    print(f"case GMRES restart {restart} refine {refine}", flush=True)
    fem, red, v, rhs, ref = _system()
    S = fem.SolverMatrix(red)
    x = torch.zeros(red.n_free, dtype=torch.float64, device="cuda")
    ws = fem.KrylovWorkspace(red.n_free, "cuda")
    before = _lib.lib().mife_gmres_cgs_refinement(refine)
    try:
        info = fem.gmres(S, S.gather(v), rhs, x, 1e-11, 20000, ws, restart=restart)
    finally:
        _lib.lib().mife_gmres_cgs_refinement(0)
    assert before == 0
    assert info.relres <= 1e-11
    # condition number below 1e3 (7 elements across, coefficients within e^+-1.5)
    assert float((x.cpu() - ref).abs().max()) <= 1e-8 * float(ref.abs().max())
    if restart >= 33:
        assert info.iterations < red.n_free


@pytest.mark.parametrize("maxit", [1, 7, 8, 9, 20])
def test_gmres_iteration_limit(maxit):
    from iron_amd import _lib
    print(f"case GMRES limit {maxit}", flush=True)
    fem, red, v, rhs, ref = _system()
    S = fem.SolverMatrix(red)
    ws = fem.KrylovWorkspace(red.n_free, "cuda")
    x = torch.zeros(red.n_free, dtype=torch.float64, device="cuda")
    with pytest.raises(_lib.NotConvergedError) as e:
        fem.gmres(S, S.gather(v), rhs, x, 1e-14, maxit, ws, restart=16)
    assert e.value.info.iterations == maxit


@pytest.mark.parametrize("fmt", ["sell", "csr"])
@pytest.mark.parametrize("f32", [False, True])
def test_minres_storages(fmt, f32):
    print(f"case MINRES {fmt} f32={f32}", flush=True)
    fem, red, v, rhs, ref = _system()
    S = fem.SolverMatrix(red, fmt)
    ws = fem.KrylovWorkspace(red.n_free, "cuda")
    x = torch.zeros(red.n_free, dtype=torch.float64, device="cuda")
    info = fem.minres(S, S.gather(v, fem.F32 if f32 else fem.F64), rhs, x, 1e-11, 20000, ws)
    assert info.iterations < red.n_free
    # condition number below 1e3, and FP32 rounding of the operator
    assert float((x.cpu() - ref).abs().max()) <= (1e-3 if f32 else 1e-8) * float(ref.abs().max())
