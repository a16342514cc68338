"""Device triangular solves of more than 64 right-hand sides: the one-launch sweeps
with products between them, and the substitution that takes over where a diagonal
block must not be inverted; against the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

EPS = {np.float64: 2.0 ** -53, np.float32: 2.0 ** -24}


def _triangle(n, upper, dtype, seed):
    r = np.random.default_rng(seed)
    t = r.standard_normal((n, n)) * (0.5 / np.sqrt(n))
    t = np.triu(t, 1) if upper else np.tril(t, -1)
    return (t + np.diag(1.0 + r.random(n))).astype(dtype), r


def _solve(a, b, upper, trans, ldb_pad=0):
    import linfa_linalg_hip as llh
    n, m = b.shape
    x = torch.full((n, m + ldb_pad), 5.0, dtype=torch.from_numpy(b).dtype, device="cuda")
    x[:, :m] = torch.from_numpy(b)
    llh.device.solve_triangular(torch.from_numpy(a).cuda(), x[:, :m],
                                llh.UPLO.Upper if upper else llh.UPLO.Lower, trans=trans)
    assert (x[:, m:] == 5.0).all()
    return x[:, :m].cpu().numpy()


@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
# one block and less; the first width of this path; ragged blocks and column
# chunks; several launches with products between them
@pytest.mark.parametrize("n,m", [(1, 65), (64, 65), (65, 100), (200, 80), (700, 129), (1000, 3100)])
def test_wide_solve(n, m, dtype, upper, trans):
    a, r = _triangle(n, upper != trans, dtype, n + m)
    b = r.standard_normal((n, m)).astype(dtype)
    x = _solve(a, b, upper, trans, ldb_pad=2)
    op = (a.T if trans else a).astype(np.float64)
    res = np.linalg.norm(op @ x.astype(np.float64) - b)
    # the residual of a substitution, gamma_n || |A| |x| ||, with a factor 4 for the
    # inverses of well-conditioned 64 x 64 blocks
    assert res <= 4 * (n + 64) * EPS[dtype] * np.linalg.norm(np.abs(op) @ np.abs(x.astype(np.float64)))


@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("n,m,i", [(100, 70, 10), (200, 100, 130)])
def test_zero_pivot_as_the_reference(n, m, i, trans):
    """A zero pivot gives the infinities and NaNs of the reference's substitution."""
    from oracle import oracle as orc
    a, r = _triangle(n, trans, np.float64, 7 * n)
    a[i, i] = 0.0
    b = r.standard_normal((n, m))
    x = _solve(a, b, False, trans)
    ref = orc.solve_triangular(np.ascontiguousarray(a.T if trans else a), b.copy(), 1)
    assert np.array_equal(np.isnan(x), np.isnan(ref)) and np.array_equal(np.isinf(x), np.isinf(ref))
    assert np.array_equal(x[i], ref[i])  # signed infinities
    assert np.allclose(x[:i], ref[:i], rtol=1e-11, atol=1e-13)


def test_ill_conditioned_block_is_substituted():
    """A block whose inverse is huge keeps the substitution's small residual."""
    n, m = 192, 80
    r = np.random.default_rng(3)
    a = np.tril(r.standard_normal((n, n)))  # condition grows exponentially with the order
    b = r.standard_normal((n, m))
    x = _solve(a, b, False, False)
    bound = 4 * n * EPS[np.float64] * np.linalg.norm(np.abs(a) @ np.abs(x))
    assert np.linalg.norm(a @ x - b) <= bound
