"""The exact-order factor and solve of small matrices with their sums in registers: the
oracle's bits at the edges of its lanes, waves and places, and its failures there."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

# one and two rows a lane (64), three in f32 (128); whole and ragged groups of places
SIZES = {np.float64: (1, 8, 9, 17, 32, 33, 63, 64, 65, 97, 127, 128),
         np.float32: (1, 31, 64, 65, 127, 128, 129, 161, 175, 176)}
CASES = [(d, n) for d in SIZES for n in SIZES[d]]


def _spd(n, dtype):
    r = np.random.default_rng(n)
    b = r.uniform(-1.0, 1.0, (n, n))
    return (b @ b.T / n + np.eye(n)).astype(dtype), r


@pytest.mark.parametrize("dtype,n", CASES)
@pytest.mark.parametrize("m", [1, 3, 8, 9, 17])
def test_bits(dtype, n, m):
    import linfa_linalg_hip as llh
    from oracle import oracle as orc
    a, r = _spd(n, dtype)
    b = r.standard_normal((n, m)).astype(dtype)
    w = torch.from_numpy(a.copy()).cuda()
    llh.device.potrf(w)
    assert np.array_equal(np.tril(w.cpu().numpy()), np.tril(orc.cholesky_dirty(a.copy())))
    f, fr = a.copy(), a.copy()
    x, xr = llh.solvec(f, b), orc.solvec(fr, b)
    assert np.array_equal(f, fr) and np.array_equal(x, xr)


@pytest.mark.parametrize("dtype,n", [c for c in CASES if c[1] > 1])
def test_failures(dtype, n):
    """Every pivot that fails is the oracle's, and so is what the factor leaves."""
    import linfa_linalg_hip as llh
    from oracle import oracle as orc
    for j in sorted({0, 1, 7, 8, 15, 16, 63, 64, n // 2, n - 2, n - 1} & set(range(n))):
        a, _ = _spd(n, dtype)
        a[j, j] = -1.0
        f, fr = a.copy(), a.copy()
        with pytest.raises(llh.NotPositiveDefinite) as e:
            llh.cholesky_inplace_dirty(f)
        with pytest.raises(Exception):
            orc.cholesky_inplace_dirty(fr)
        assert e.value.column == j and np.array_equal(f, fr)
