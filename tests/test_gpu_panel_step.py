"""The one-launch panel step of the blocked factor (device potrf) at the edges of
its blocks, panels and failure handling, against LAPACK's factor in float64."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

EPS = {torch.float64: 2.0 ** -53, torch.float32: 2.0 ** -24}


def _spd(n, dtype, seed):
    r = np.random.default_rng(seed)
    b = r.standard_normal((n, n))
    return torch.from_numpy(b @ b.T / n + np.eye(n)).to(dtype)


@pytest.mark.parametrize("pad", [0, 3])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
# one block more than the exact kernel takes; ragged and whole last blocks; the
# widest single panel and the first order with a panel before it
@pytest.mark.parametrize("n", [177, 191, 192, 193, 256, 577, 1089, 4096, 4097, 4161])
def test_potrf_block_edges(n, dtype, pad):
    import linfa_linalg_hip as llh
    a = _spd(n, dtype, n)
    w = torch.full((n, n + pad), 7.0, dtype=dtype, device="cuda")
    low = torch.tril(a).cuda()
    w[:, :n] = low + torch.triu(torch.full((n, n), float("nan"), dtype=dtype, device="cuda"), 1)
    llh.device.potrf(w[:, :n])
    l = torch.tril(w[:, :n]).double()
    full = low.double() + torch.tril(low.double(), -1).T
    # backward error of a Cholesky factor: gamma_(n+1) || |L| |L^T| ||_F, and
    # || |L| |L^T| ||_F <= sqrt(n) ||A||_F for a matrix of this norm
    err = (full - l @ l.T).norm() / full.norm()
    assert err <= (n + 1) * EPS[dtype], float(err)
    # the strict upper triangle and the padding are untouched
    assert torch.isnan(w[:, :n][torch.triu(torch.ones(n, n, device="cuda"), 1) > 0]).all()
    assert (w[:, n:] == 7.0).all()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n,f", [(300, 0), (300, 15), (300, 16), (300, 63), (300, 64), (300, 200), (300, 256),
                                 (300, 299), (700, 383), (700, 384)])
def test_potrf_failure_rows(n, f, dtype):
    """Rows before the failing one hold L, the failing row L[f, ..f], and the plain
    form leaves the rest of the array as it was."""
    import linfa_linalg_hip as llh
    a = _spd(n, torch.float64, n + f)
    l = torch.linalg.cholesky(a)
    a[f, f] = (l[f, :f] ** 2).sum() - 0.5
    w = a.to(dtype).cuda()
    with pytest.raises(llh.NotPositiveDefinite) as e:
        llh.device.potrf(w)
    assert e.value.column == f
    tol = 8 * (n + 1) * EPS[dtype]  # forward error: the leading block has condition < 8
    got = torch.tril(w[:f, :f]).double().cpu()
    assert (got - l[:f, :f]).norm() <= tol * max(1.0, l[:f, :f].norm())
    assert (w[f, :f].double().cpu() - l[f, :f]).norm() <= tol * max(1.0, l[f, :f].norm())
    host = a.to(dtype).numpy().copy()
    ref = host.copy()
    with pytest.raises(llh.NotPositiveDefinite):
        llh.cholesky_inplace_dirty(host)
    assert np.array_equal(host[f + 1:], ref[f + 1:]) and np.array_equal(host[f, f:], ref[f, f:])
    assert np.array_equal(np.triu(host, 1), np.triu(ref, 1))
