"""The device inverse at the edges of its levels of blocks, against LAPACK in float64."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

EPS = {torch.float64: 2.0 ** -53, torch.float32: 2.0 ** -24}


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
# three blocks (a pair and a single one), a power of two of blocks, one row more,
# a last block of one row in the second half of a large pair
@pytest.mark.parametrize("n", [177, 192, 256, 257, 321, 1025])
@pytest.mark.parametrize("pad", [0, 5])
def test_inverse_levels(n, pad, dtype):
    import linfa_linalg_hip as llh
    r = np.random.default_rng(n)
    b = r.standard_normal((n, n))
    a = torch.from_numpy(b @ b.T / n + np.eye(n)).to(dtype)
    w = a.cuda()
    out = torch.full((n, n + pad), 3.0, dtype=dtype, device="cuda")
    llh.device.invc(w, out[:, :n])
    x = out[:, :n].double().cpu()
    assert torch.equal(x, x.T)  # one product gives both triangles
    assert (out[:, n:] == 3.0).all()
    # || A X - I || <= c n eps cond(A) with cond(A) < 6 for this construction
    res = (a.double() @ x - torch.eye(n, dtype=torch.float64)).norm()
    assert res <= 6 * n * EPS[dtype] * np.sqrt(n), float(res)
