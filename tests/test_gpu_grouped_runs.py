"""Grouped CG in runs of any length: the FP64 iterates of a segment depend neither on
where the runs of iterations end nor on how often a group looks for FP32 replacements,
and agree with the single solve.  Sizes below, at and beyond what a block of the product
and of the update takes (SELL3: 64 and 256 node rows; SELL: 256 and 1024 rows) and beyond
the 384 update blocks whose partial sums a product block holds in registers."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# free rows: diffusion (nx - 1)(ny + 1)(nz + 1), elasticity nodes nx (ny + 1)(nz + 1)
CASES = [("diffusion", (2, 1, 1), 2e8), ("diffusion", (17, 3, 3), 2e8), ("diffusion", (34, 5, 5), 2e8),
         ("diffusion", (75, 74, 73), 2e9), ("elasticity", (1, 1, 1), 2e8), ("elasticity", (16, 1, 1), 2e8),
         ("elasticity", (13, 4, 3), 2e8), ("elasticity", (16, 3, 3), 2e8)]


def _serve(reqs, budget, **options):
    from iron_amd import serving
    srv = serving.Server(hbm_budget=budget, max_segments=8, **options)
    return {r.rid: r for r in srv.run(reqs)}


@pytest.mark.parametrize("kind,ne,budget", CASES)
def test_runs_of_any_length_give_the_same_iterates(kind, ne, budget):
    from iron_amd import serving
    print(f"case grouped runs {kind} {ne}", flush=True)

    def req():
        return serving.Request(0, kind, ne, 21, rtol=1e-11)

    ref = _serve([req()], budget, precision="fp64", chunk=16)[0]
    for chunk in (1, 7):
        r = _serve([req()], budget, precision="fp64", chunk=chunk)[0]
        assert r.iterations == ref.iterations
        assert np.array_equal(r.u, ref.u), chunk
    # two solves to 1e-11 of systems with condition numbers up to 1e5
    one = serving.solve_one_fp64(req(), {})
    assert np.abs(ref.u - one.u).max() <= 1e-6 * max(1.0, np.abs(one.u).max())


def test_fp64_segment_next_to_mixed_ones():
    from iron_amd import serving
    print("case grouped runs: FP64 next to mixed", flush=True)

    def reqs():
        return [serving.Request(0, "diffusion", (9, 7, 6), 31), serving.Request(1, "elasticity", (7, 4, 3), 32)]

    fp64 = _serve(reqs(), 2e8, precision="fp64", chunk=16)
    split = _serve(reqs(), 2e8, precision="split", chunk=16)
    kept = [k for k, r in fp64.items() if r.kind not in serving.Server.MIXED_KINDS["split"]]
    assert len(kept) == 1
    for k in kept:
        assert split[k].iterations == fp64[k].iterations and np.array_equal(split[k].u, fp64[k].u)


@pytest.mark.parametrize("ne", [(67, 39, 39), (68, 39, 39), (40, 39, 38), (40, 39, 39)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_elasticity_with_a_slice_per_wavefront(ne, precision):
    """Slice counts below and at those from which a block's wavefronts take a SELL3 slice
    each: 1,700 (FP64) and 1,000 (FP32), nodes nx (ny + 1)(nz + 1) in slices of 64."""
    from iron_amd import serving
    print(f"case grouped SELL3 {ne} {precision}", flush=True)

    def req():
        return serving.Request(0, "elasticity", ne, 17, rtol=1e-9)

    ref = _serve([req()], 2e9, precision=precision, chunk=16)[0]
    one = serving.solve_one_fp64(req(), {})
    # two solves to 1e-9 of systems with condition numbers up to 1e5
    assert np.abs(ref.u - one.u).max() <= 1e-4 * np.abs(one.u).max()
    if precision == "fp64":
        other = _serve([req()], 2e9, precision=precision, chunk=7)[0]
        assert other.iterations == ref.iterations and np.array_equal(other.u, ref.u)


def test_streamed_segments_beside_kept_ones():
    """A group beyond what the cache keeps (the first two diffusion requests fit it, the
    third and the elasticity one do not): every solution is that of the request served
    alone, where it is kept, bit for bit."""
    from iron_amd import serving
    print("case grouped runs: kept and streamed segments", flush=True)

    def reqs():
        return [serving.Request(k, kind, ne, 40 + k, rtol=1e-8) for k, (kind, ne) in enumerate([
            ("diffusion", (65, 74, 73)), ("diffusion", (66, 60, 73)), ("diffusion", (75, 74, 73)),
            ("elasticity", (40, 24, 22))])]

    both = _serve(reqs(), 8e9, precision="fp64", chunk=16)
    for r in reqs():
        alone = _serve([r], 8e9, precision="fp64", chunk=16)[r.rid]
        assert alone.iterations == both[r.rid].iterations and np.array_equal(alone.u, both[r.rid].u), r.rid
