"""Products far smaller than what they are subtracted from are summed first: each alone
would be lost in the rounding, their sum is not.  All values are powers of two, so the
expected entries are exact."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pad", [0, 3])
# columns summed: one panel step's 64 (f64), two steps' 128 (f32); rows to n = 320 and to
# more than a workgroup row of tiles
@pytest.mark.parametrize("dtype,cols", [(torch.float64, 64), (torch.float32, 128)])
@pytest.mark.parametrize("n", [320, 1000])
def test_updates_of_later_columns(n, dtype, cols, pad):
    """Column 192, whose entries of 1 lose the products of the first columns."""
    import linfa_linalg_hip as llh
    # u v is below half an ulp of 1 even for a quarter of the columns; cols u v is an ulp or more
    u, v = (2.0 ** -28, 2.0 ** -28) if dtype == torch.float64 else (2.0 ** -15, 2.0 ** -16)
    a = torch.eye(n, dtype=torch.float64)
    a[193:, 193:] *= 100.0 * n
    a[192, :cols], a[193:, :cols] = u, v
    a[192, 192], a[193:, 192] = 1.0 + cols * u * u, 1.0
    w = torch.zeros(n, n + pad, dtype=dtype, device="cuda")
    w[:, :n] = a.to(dtype)
    llh.device.potrf(w[:, :n])
    l = w[:, 192].double().cpu()
    assert l[192] == 1.0
    assert (l[193:] == 1.0 - cols * u * v).all()


@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("dtype,t", [(np.float64, 2.0 ** -28), (np.float32, 2.0 ** -14)])
def test_substitution(dtype, t, upper):
    """Rows of 1 from which a block of 16 columns takes 16 t^2 = 2^-52 (2^-24)."""
    import linfa_linalg_hip as llh
    n, m = 64, 70
    a = np.eye(n, dtype=dtype)
    b = np.ones((n, m), dtype=dtype)
    a[16:, :16] = t
    b[:16] = t
    if upper:
        a, b = np.ascontiguousarray(a[::-1, ::-1]), np.ascontiguousarray(b[::-1])
    x = torch.from_numpy(b).cuda()
    llh.device.solve_triangular(torch.from_numpy(a).cuda(), x, llh.UPLO.Upper if upper else llh.UPLO.Lower)
    x = x.cpu().numpy()[::-1 if upper else 1]
    assert (x[:16] == t).all() and (x[16:] == 1.0 - 16.0 * t * t).all()
