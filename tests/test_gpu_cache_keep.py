"""Products of a matrix part of which is read with plain loads (kept in the Infinity
Cache between products) and part of which is streamed: the split follows the stored size
a descriptor states and changes how values are loaded, never what is added, so a
product is the same bit for bit at every split.  The stated size is raised on small
matrices to reach the partial splits (all, some sixteenths, none)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["sell16", "sell32", "sell3"])
@pytest.mark.parametrize("schedule", [True, False])
def test_products_do_not_depend_on_the_kept_part(fmt, schedule):
    from iron_amd import _lib, basis, fem, mesh
    ncomp = 3 if fmt == "sell3" else 1
    ne = (19, 17, 13)
    b = basis.basis(3, 1)
    m = mesh.RegularMesh(ne, [b], (1.0, 1.0, 1.0))
    dm = mesh.DofMap(m, [0] * ncomp)
    csr = fem.CSRStructure(dm.element_dofs(), dm.num_dofs, colours=mesh.structured_colours(m))
    red = fem.DirichletReduction(csr, np.tile(m.coords[:, 0] == 0.0, ncomp))
    S = fem.SolverMatrix(red, compress=fmt != "sell32", schedule=schedule,
                         interleave=(3, m.num_nodes(0)) if ncomp == 3 else None, block=ncomp == 3)
    assert (S.fmt == "sell3") == (fmt == "sell3") and (S.col16 is None) == (fmt == "sell32")
    g = torch.Generator(device="cuda").manual_seed(3)
    v = torch.randn(csr.nnz, dtype=torch.float64, device="cuda", generator=g)
    for prec, dt in ((fem.F64, torch.float64), (fem.F32, torch.float32)):
        vals = S.gather(v, prec)
        x = torch.randn(S.n, dtype=dt, device="cuda", generator=g)
        want, stored = None, S.desc.nnz
        for nnz in (stored, 25_000_000, 40_000_000, 200_000_000, 10_000_000_000):
            print(f"case {fmt} schedule={schedule} prec={prec} stated entries {nnz}", flush=True)
            S.desc.nnz = nnz
            y = S.spmv(vals, x, torch.full((S.n,), float("nan"), dtype=dt, device="cuda"), prec)
            torch.cuda.synchronize()
            want = y if want is None else want
            assert torch.equal(y, want) and bool(torch.isfinite(y).all())
        S.desc.nnz = stored
    # the products above against CSR (FP64)
    Sc = fem.SolverMatrix(red, "csr")
    x0 = torch.randn(red.n_free, dtype=torch.float64, device="cuda", generator=g)
    perm = S.perm.long()
    y = torch.empty_like(x0)
    y[perm] = S.spmv(S.gather(v), x0[perm].contiguous(), torch.empty_like(x0))
    ref = Sc.spmv(Sc.gather(v), x0, torch.empty_like(x0))
    # both are FP64 sums of at most 81 products in different orders
    assert float((y - ref).abs().max()) <= 1e-13 * 81 * float(ref.abs().max())
