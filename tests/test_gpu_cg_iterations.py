"""Jacobi CG stopped by its iteration limit, at limits around the solver's chunk
lengths (an iteration hands its scalars from one state slot to the other, a chunk
ends in a finisher): the iterate equals that of the textbook recurrence after as many
iterations, FP64, on scheduled and unscheduled SELL, SELL3 and CSR storage, with
and without graph replay."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _textbook(A, b, k):
    """x after k iterations of Jacobi-preconditioned CG from zero (FP64, host)."""
    d = A.diagonal()
    x, r = np.zeros_like(b), b.copy()
    z = r / d
    p = z.copy()
    rz = r @ z
    for _ in range(k):
        q = A @ p
        alpha = rz / (p @ q)
        x += alpha * p
        r -= alpha * q
        z = r / d
        rz, old = r @ z, rz
        p = z + (rz / old) * p
    return x


@pytest.mark.parametrize("storage", ["sell", "sell-plain", "csr", "sell3"])
@pytest.mark.parametrize("graphs", [True, False])
def test_limited_iterations_match_the_textbook_recurrence(storage, graphs):
    import scipy.sparse as sp
    from iron_amd import _lib, basis, fem, mesh
    ncomp = 3 if storage == "sell3" else 1
    b = basis.basis(3, 1)
    m = mesh.RegularMesh((11, 7, 9), [b], (1.0, 1.0, 1.0))
    dm = mesh.DofMap(m, [0] * ncomp)
    csr = fem.CSRStructure(dm.element_dofs(), dm.num_dofs, colours=mesh.structured_colours(m))
    g = torch.Generator(device="cuda").manual_seed(5)
    E = m.num_elements
    z = torch.randn(E, dtype=torch.float64, device="cuda", generator=g).mul(0.3).exp()
    v = csr.zeros()
    if ncomp == 1:
        fem.ScalarAssembler(b, m.coords, m.elem_nodes[0], csr).assemble(v, kappa=z)
    else:
        nu = torch.full_like(z, 0.3)
        fem.ElasticAssembler(b, m.coords, m.elem_nodes[0], csr).assemble(v, torch.stack([z, z, z, nu, nu, nu], dim=1))
    red = fem.DirichletReduction(csr, np.tile(m.coords[:, 0] == 0.0, ncomp))
    S = fem.SolverMatrix(red, "csr" if storage == "csr" else "sell", schedule=storage != "sell-plain",
                         interleave=(3, m.num_nodes(0)) if ncomp == 3 else None, block=ncomp == 3)
    assert (S.fmt == "sell3") == (storage == "sell3")
    kv = red.gather(v).cpu().numpy()
    A = sp.csr_matrix((kv, red.col[: red.nnz].cpu().numpy(), red.row_ptr.cpu().numpy()))
    bvec = torch.randn(red.n_free, dtype=torch.float64, device="cuda", generator=g)
    ws = fem.KrylovWorkspace(red.n_free, "cuda")
    vals = S.gather(v)
    _lib.graphs_enable(graphs)
    try:
        for k in (1, 2, 7, 8, 9, 15, 16, 17, 24):
            print(f"case {storage} graphs={graphs} limit {k}", flush=True)
            x = torch.zeros_like(bvec)
            with pytest.raises(_lib.NotConvergedError) as e:
                fem.cg(S, vals, bvec, x, 1e-30, k, ws)
            assert e.value.info.iterations == k
            want = _textbook(A, bvec.cpu().numpy(), k)
            # two FP64 recurrences in different summation orders: rounding (about n eps per
            # step in the dot products) grows with the steps taken, far below 1e-10 here
            assert np.abs(x.cpu().numpy() - want).max() <= 1e-10 * np.abs(want).max()
    finally:
        _lib.graphs_enable(True)
