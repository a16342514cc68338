"""A panel step whose block fails: no workgroup of its launch finds the block changed by
another one, so the block keeps its entries beyond the failing row and every entry of
the array is the same from call to call."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def _failing(n, f, dtype):
    r = np.random.default_rng(n + f)
    b = r.standard_normal((n, n))
    a = torch.from_numpy(b @ b.T / n + np.eye(n))
    l = torch.linalg.cholesky(a[:f, :f])
    row = torch.linalg.solve_triangular(l, a[:f, f:f + 1], upper=False)
    a[f, f] = (row ** 2).sum() - 0.5
    return a.to(dtype).cuda()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n,f", [(300, 16), (300, 40), (1000, 62), (2500, 33)])
def test_first_block_beyond_the_failing_row(n, f, dtype):
    import linfa_linalg_hip as llh
    a = _failing(n, f, dtype)
    w = a.clone()
    with pytest.raises(llh.NotPositiveDefinite) as e:
        llh.device.potrf(w)
    assert e.value.column == f
    assert torch.equal(w[f + 1:64, :64], a[f + 1:64, :64]) and w[f, f] == a[f, f]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n,f", [(700, 300), (2500, 20), (2500, 700), (2500, 2490)])
def test_the_same_from_call_to_call(n, f, dtype):
    import linfa_linalg_hip as llh
    a = _failing(n, f, dtype)
    first = None
    for _ in range(4):
        w = a.clone()
        with pytest.raises(llh.NotPositiveDefinite) as e:
            llh.device.potrf(w)
        assert e.value.column == f
        first = w if first is None else first
        assert torch.equal(w, first)
