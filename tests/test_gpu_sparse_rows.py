"""Back-substitution and the lifted RHS on CSR matrices of ragged rows (empty ones, one
entry, more entries in a block's rows than a tile holds, row counts around the rows per
block), against host sums.  Both sides add a row's products in FP64 in different
orders: the bound is the row length times eps times the sum of the products' magnitudes."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _matrix(n, lengths, rng):
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in lengths] + [np.zeros(0)]).astype(np.int32)
    return rp, col, rng.standard_normal(rp[-1])


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


@pytest.mark.parametrize("n,kind", [(1, "full"), (31, "ragged"), (32, "ragged"), (33, "ragged"), (257, "empty"),
                                    (300, "full"), (2600, "long"), (1030, "ragged")])
def test_backsubstitution_and_rhs_rows(n, kind):
    from iron_amd import _lib
    print(f"case n={n} rows={kind}", flush=True)
    rng = np.random.default_rng(n)
    lengths = {"full": np.full(n, n), "ragged": rng.integers(0, min(n, 130) + 1, n), "empty": np.zeros(n, int),
               "long": np.where(rng.random(n) < 0.02, n, rng.integers(0, 90, n))}[kind]
    rp, col, vals = _matrix(n, lengths, rng)
    u, src, rhs = (rng.standard_normal(n) for _ in range(3))
    u[rng.random(n) < 0.2] = 0.0
    fixed_row = (rng.random(n) < 0.25).astype(np.uint8)
    d = [_dev(a) for a in (rp, col if len(col) else np.zeros(1, np.int32), vals if len(vals) else np.zeros(1), u, src)]
    R = torch.empty(n, dtype=torch.float64, device="cuda")
    rows = np.repeat(np.arange(n), lengths)
    inrow = np.arange(len(col)) - rp[rows]
    for compat in (0, 1):
        for flags in (None, fixed_row):
            fl = None if flags is None else _dev(flags)
            _lib.call("mife_backsubstitute", n, *[_lib.ptr(t) for t in d], _lib.ptr(fl), compat, _lib.ptr(R), None)
            prod = vals * u[inrow if compat else col]
            if flags is not None:
                prod = np.where(flags[rows] != 0, 0.0, prod)
            want = np.bincount(rows, prod, n) - src
            lim = EPS * (np.maximum(lengths, 1) + 2) * (np.bincount(rows, np.abs(prod), n) + np.abs(src))
            assert np.all(np.abs(R.cpu().numpy() - want) <= lim)
    # lifted RHS over the free DOFs, rows flagged in fixed_row without lifting
    free = np.nonzero(rng.random(n) < 0.6)[0].astype(np.int32)
    if len(free) == 0:
        free = np.zeros(1, np.int32)
    new_idx = np.full(n, -1, np.int32)
    new_idx[free] = np.arange(len(free))
    b = torch.empty(len(free), dtype=torch.float64, device="cuda")
    for flags in (None, fixed_row):
        fl = None if flags is None else _dev(flags)
        args = [_dev(free), d[0], d[1], d[2], _dev(new_idx), d[3], d[4], _dev(rhs)]
        _lib.call("mife_solver_rhs", len(free), *[_lib.ptr(t) for t in args], _lib.ptr(fl), _lib.ptr(b), None)
        prod = np.where(new_idx[col] < 0, -vals * u[col], 0.0)
        if flags is not None:
            prod = np.where(flags[rows] != 0, 0.0, prod)
        want = (src + rhs + np.bincount(rows, prod, n))[free]
        lim = EPS * ((np.maximum(lengths, 1) + 3) * (np.bincount(rows, np.abs(prod), n) + np.abs(src) + np.abs(rhs)))[free]
        assert np.all(np.abs(b.cpu().numpy() - want) <= lim)


@pytest.mark.parametrize("n", [16383, 16384, 16385, 40001])
def test_backsubstitution_rows_per_block(n):
    """Row counts about the one from which a block takes 32 rows instead of 16; rows of 0 to
    140 entries, so that blocks hold less than a tile, about one and more than two."""
    from iron_amd import _lib
    print(f"case n={n}", flush=True)
    rng = np.random.default_rng(n)
    lengths = np.where(np.arange(n) // 500 % 2 == 0, rng.integers(0, 30, n), rng.integers(50, 141, n))
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    rows = np.repeat(np.arange(n), lengths)
    inrow = np.arange(rp[-1]) - rp[rows]
    col = ((rows + 17 * inrow) % n).astype(np.int32)
    vals, u, src = rng.standard_normal(rp[-1]), rng.standard_normal(n), rng.standard_normal(n)
    fixed = (rng.random(n) < 0.25).astype(np.uint8)
    d = [_dev(a) for a in (rp, col, vals, u, src, fixed)]
    R = torch.empty(n, dtype=torch.float64, device="cuda")
    for compat in (0, 1):
        _lib.call("mife_backsubstitute", n, *[_lib.ptr(t) for t in d], compat, _lib.ptr(R), None)
        prod = np.where(fixed[rows] != 0, 0.0, vals * u[inrow if compat else col])
        want = np.bincount(rows, prod, n) - src
        lim = EPS * (lengths + 3) * (np.bincount(rows, np.abs(prod), n) + np.abs(src))
        assert np.all(np.abs(R.cpu().numpy() - want) <= lim)
