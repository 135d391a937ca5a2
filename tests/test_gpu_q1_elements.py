"""Trilinear element kernels (eight elements per wavefront, 32 per block) at element
counts around those numbers, on moved nodes: the structured, coloured and atomic
assemblies against the oracle's element matrices, scalar with a source and elasticity,
FP64 and FP32.  FP64 tolerance: 1e-13 of the largest entry (sums of 24 products in
another order, geometry through an explicit inverse); FP32 2e-6 (24 roundings of 6e-8)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from oracle import fe_oracle as fo  # noqa: E402


@pytest.mark.parametrize("ne", [(1, 1, 1), (7, 1, 1), (2, 2, 2), (9, 1, 1), (31, 1, 1), (4, 4, 2), (33, 1, 1),
                                (13, 5, 1)])
@pytest.mark.parametrize("ncomp", [1, 3])
def test_q1_elements_match_oracle(ne, ncomp):
    from iron_amd import basis, fem, mesh
    b = basis.basis(3, 1)
    m = mesh.RegularMesh(ne, [b], (1.0, 1.2, 0.9))
    dm = mesh.DofMap(m, [0] * ncomp)
    rng = np.random.default_rng(sum(ne) + ncomp)
    h = np.array([1.0, 1.2, 0.9]) / np.array(ne)
    X = m.coords + 0.1 * h * (rng.random(m.coords.shape) - 0.5)
    E = m.num_elements
    ob = fo.Basis(3, 1, 2)
    om = fo.regular_mesh(ne, [ob], (1.0, 1.2, 0.9))
    od = fo.DofMap(om, [0] * ncomp)
    xe = X[om.elem_nodes[0] - 1]
    rp, col = fo.csr_pattern(od)
    coef = np.exp(rng.standard_normal(E))
    if ncomp == 1:
        Ke = fo.laplace_element_matrices(xe, ob, coef)
        src = rng.standard_normal(E)
        sref = fo.assemble_vector(od.element_dofs(), fo.poisson_source_vectors(xe, ob, src), od.num_dofs)
        coef_d = torch.as_tensor(coef, device="cuda")
    else:
        mat = np.stack([10 * coef, 9 * coef, 11 * coef] + [np.full(E, v) for v in (0.3, 0.28, 0.31)], axis=1)
        Ke = fo.linear_elasticity_element_matrices(xe, ob, fo.linear_elasticity_tensor(*mat.T))
        coef_d = torch.as_tensor(np.ascontiguousarray(mat), device="cuda")
    ref = fo.assemble_csr(rp, col, od.element_dofs(), Ke, od.num_dofs)
    for form in ("structured", "coloured", "atomic"):
        csr = fem.CSRStructure(dm.element_dofs(), dm.num_dofs, colours=mesh.structured_colours(m))
        grid = ne if form == "structured" else None
        for prec, tol in ((fem.F64, 1e-13), (fem.F32, 2e-6)):
            print(f"case {ne} components={ncomp} {form} prec={prec}", flush=True)
            v = csr.zeros(prec)
            s = torch.zeros(csr.n, dtype=torch.float64, device="cuda")
            if ncomp == 1:
                asm = fem.ScalarAssembler(b, X, m.elem_nodes[0], csr, grid=grid)
                asm.assemble(v, kappa=coef_d, source=torch.as_tensor(src, device="cuda"), src_vec=s, prec=prec,
                             atomic=form == "atomic")
                assert np.abs(s.cpu().numpy() - sref).max() <= 1e-13 * np.abs(sref).max()
            else:
                fem.ElasticAssembler(b, X, m.elem_nodes[0], csr, grid=grid).assemble(v, coef_d, prec=prec,
                                                                                     atomic=form == "atomic")
            assert np.abs(v[: csr.nnz].cpu().numpy() - ref).max() <= tol * np.abs(ref).max()
