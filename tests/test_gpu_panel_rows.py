"""The rows below a panel's top block (one launch for all of the panel's columns) at the
edges of its strips, in every storage and arithmetic type, against the matrix itself."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

EPS = {torch.float64: 2.0 ** -53, torch.float32: 2.0 ** -24}


def _spd(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    b = torch.randn(n, n, dtype=torch.float64, device="cuda", generator=g)
    a = b @ b.T / n
    a.diagonal().add_(1.0)
    return a


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
# the first orders with such rows (one more than the panels stepped through whole; a
# strip of one row, a whole one), more strips than CUs, and rows not a multiple of 16
# bytes apart
@pytest.mark.parametrize("n,pad", [(8193, 0), (8224, 0), (8225, 7), (9000, 3), (17409, 0)])
def test_potrf_rows_below(n, pad, dtype):
    import linfa_linalg_hip as llh
    a = _spd(n, n).to(dtype)
    w = torch.full((n, n + pad), 7.0, dtype=dtype, device="cuda")
    w[:, :n] = torch.tril(a)
    llh.device.potrf(w[:, :n])
    l = torch.tril(w[:, :n]).double()
    # backward error of a Cholesky factor: gamma_(n+1) || |L| |L^T| ||_F, and
    # || |L| |L^T| ||_F <= sqrt(n) ||A||_F for a matrix of this norm
    err = (a.double() - l @ l.T).norm() / a.double().norm()
    assert err <= (n + 1) * EPS[dtype], float(err)
    assert (torch.triu(w[:, :n], 1) == 0).all() and (w[:, n:] == 7.0).all()


@pytest.mark.parametrize("f", [0, 63, 64, 300, 511, 512, 700])
def test_failure_in_the_top_block(f):
    """A failure among the columns of a top block stops the rows below it too."""
    import linfa_linalg_hip as llh
    n = 8300
    a = _spd(n, f)
    l = torch.linalg.cholesky(a[: f + 1, : f + 1])
    a[f, f] = (l[f, :f] ** 2).sum() - 0.5
    w = a.clone()
    with pytest.raises(llh.NotPositiveDefinite) as e:
        llh.device.potrf(w)
    assert e.value.column == f
    tol = 8 * (n + 1) * EPS[torch.float64]  # forward error: condition < 8
    got = torch.tril(w[: f + 1, : f + 1])
    assert (got[:f, :f] - l[:f, :f]).norm() <= tol * max(1.0, float(l.norm()))
    assert (got[f, :f] - l[f, :f]).norm() <= tol * max(1.0, float(l.norm()))


@pytest.mark.parametrize("prec", ["f32", "f16"])
def test_refined_solve(prec):
    """The refinement solve's factors (f64 diagonal blocks, f16 updates)."""
    import linfa_linalg_hip as llh
    n = 8300
    a = _spd(n, 5)
    x = torch.randn(n, 3, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(6))
    out = torch.empty_like(x)
    rhs = a @ x
    llh.device.solve_mixed(a, rhs, out, prec=prec)
    # the refinement stops at a float64 backward error; condition < 8
    assert (out - x).norm() <= 8 * n * EPS[torch.float64] * x.norm()
