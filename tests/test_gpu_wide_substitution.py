"""Solves with more than 64 right-hand sides are substitutions, row by row: the residual
of each row stays that of a substitution whatever the condition of a 64 x 64 diagonal
block, and infinities and NaNs reach the rows that the reference's sweep
(triangular.rs:113-125) carries them to, and no other."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

EPS = {np.float64: 2.0 ** -53, np.float32: 2.0 ** -24}
FORMS = [(False, False), (True, False), (False, True), (True, True)]


def _solve(a, b, upper, trans):
    import linfa_linalg_hip as llh
    x = torch.from_numpy(b).cuda()
    llh.device.solve_triangular(torch.from_numpy(a).cuda(), x, llh.UPLO.Upper if upper else llh.UPLO.Lower,
                                trans=trans)
    return x.cpu().numpy()


def _stored(op, upper, trans):
    """The array whose (transposed) triangle is op, the other triangle filled with NaN."""
    a = op.T if trans else op
    return np.where(np.triu(np.ones_like(a)) > 0 if upper != trans else np.tril(np.ones_like(a)) > 0, a,
                    np.nan).astype(op.dtype)


def _growing(n, c, dtype, seed):
    """Unit lower triangle, -c below: the inverse of a 64 x 64 block grows as (1 + c)^64."""
    r = np.random.default_rng(seed)
    return (np.tril(-c * (1 + 0.05 * r.random((n, n))), -1) + np.eye(n)).astype(dtype), r


def _worst(op, x, b):
    """max over the entries of |b - op x| / (|op| |x|), in longer arithmetic"""
    op, x = op.astype(np.longdouble), x.astype(np.longdouble)
    return float((np.abs(b - op @ x) / (np.abs(op) @ np.abs(x))).max())


@pytest.mark.parametrize("upper,trans", FORMS)
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
# one block; whole and ragged ones.  max |M| max |M^-1| of a block: 2.6e2, 2.9e3, 5.3e3
@pytest.mark.parametrize("n,c", [(64, 0.13), (64, 0.17), (200, 0.17), (200, 0.18)])
def test_rows_of_ill_conditioned_blocks(n, c, dtype, upper, trans):
    op, r = _growing(n, c, dtype, n)
    if upper:
        op = np.ascontiguousarray(op[::-1, ::-1])
    b = (op.astype(np.float64) @ r.standard_normal((n, 80))).astype(dtype)
    x = _solve(_stored(op, upper, trans), b, upper, trans)
    # every row of a substitution: gamma_n, with a factor (1 + eps)^2 for the pivots' reciprocals
    assert _worst(op, x, b) <= (n + 4) * EPS[dtype]


@pytest.mark.parametrize("form", ["device", "noalloc", "host"])
def test_solve_of_an_ill_conditioned_system(form):
    """Both substitutions after the factor, against L L^T with the factor as it is."""
    import linfa_linalg_hip as llh
    from linfa_linalg_hip import _abi
    n, m = 200, 80
    t, r = _growing(n, 0.15, np.float64, 3)
    for i in range(0, n, 64):
        t[i + 64:, i:i + 64] *= 0.002
    a = t @ t.T
    b = a @ r.standard_normal((n, m))
    if form == "host":
        w = a.copy()
        x = llh.solvec(w, b)
    else:
        w, x = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
        if form == "device":
            llh.device.solvec(w, x)
        else:
            c, err = llh.device.context(), _abi.LlhError()
            assert c._lib.llh_dev_solvec_noalloc_d(c.handle, n, ctypes.c_void_p(w.data_ptr()), n, m,
                                                   ctypes.c_void_p(x.data_ptr()), m, ctypes.byref(err)) == 0
        w, x = w.cpu().numpy(), x.cpu().numpy()
    l = np.tril(w).astype(np.longdouble)
    x = x.astype(np.longdouble)
    worst = np.abs(b - l @ (l.T @ x)) / (np.abs(l) @ (np.abs(l.T) @ np.abs(x)))
    assert float(worst.max()) <= 2 * (n + 4) * EPS[np.float64]


@pytest.mark.parametrize("upper,trans", FORMS)
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("what", ["b_inf", "b_nan", "a_block", "a_tile", "pivot_inf", "pivot_nan", "pivot_zero"])
def test_infinities_and_nans_as_the_reference(what, dtype, upper, trans):
    from oracle import oracle as orc
    n, m, i = 200, 70, 100  # row i lies in the second block, in solve order too
    r = np.random.default_rng(5)
    op = r.standard_normal((n, n)) * (0.5 / np.sqrt(n))
    op = np.triu(op, 1) if upper else np.tril(op, -1)
    op = (op + np.diag(1.0 + r.random(n))).astype(dtype)
    b = r.standard_normal((n, m)).astype(dtype)
    near, far = (i + 5, n - 3) if upper else (i - 5, 3)  # solved before row i: in its block, in another
    if what == "b_inf":
        b[i, ::3] = np.inf
        b[i, 1::3] = -np.inf
    elif what == "b_nan":
        b[i, 7] = b[i, 69] = np.nan
    elif what == "a_block":
        op[i, near] = np.inf
    elif what == "a_tile":
        op[i, far] = np.inf
    else:
        op[i, i] = {"pivot_inf": np.inf, "pivot_nan": np.nan, "pivot_zero": 0.0}[what]
    x = _solve(_stored(op, upper, trans), b, upper, trans)
    ref = orc.solve_triangular(np.ascontiguousarray(op), b.copy(), 0 if upper else 1)
    assert np.array_equal(np.isnan(x), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(np.isinf(x), inf) and np.array_equal(x[inf], ref[inf])
    fin = np.isfinite(ref)
    # condition < 8, rows of ordinary size
    assert np.abs(x[fin] - ref[fin]).max() <= 8 * (n + 4) * EPS[dtype] * np.abs(ref[fin]).max()


@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_pivots_without_a_normal_reciprocal(dtype, upper):
    """Subnormal pivots and pivots near the largest number are divided by."""
    n, m = 130, 66
    fi = np.finfo(dtype)
    r = np.random.default_rng(9)
    op = r.standard_normal((n, n)) * 0.05
    op = np.triu(op, 1) if upper else np.tril(op, -1)
    op = (op + np.diag(1.0 + r.random(n))).astype(dtype)
    b = r.standard_normal((n, m)).astype(dtype)
    x0 = r.uniform(1, 2, m).astype(dtype)
    for i, d in ((20, fi.smallest_subnormal * dtype(8)), (70, fi.max / dtype(4)), (128, fi.tiny / dtype(16))):
        # (the row is the pivot's alone: its x is about x0 and of use to later rows)
        op[i, :] = 0
        op[i, i] = d
        b[i] = d * x0
    x = _solve(_stored(op, upper, False), b, upper, False)
    for i in (20, 70, 128):
        assert np.array_equal(x[i], b[i] / op[i, i])  # one division
    ordinary = [k for k in range(n) if k not in (20, 70, 128)]
    o, y = op.astype(np.longdouble), x.astype(np.longdouble)
    worst = (np.abs(b - o @ y) / (np.abs(o) @ np.abs(y)))[ordinary]
    assert float(worst.max()) <= (n + 4) * EPS[dtype]
