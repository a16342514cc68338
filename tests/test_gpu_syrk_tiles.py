"""The large trailing updates of the blocked factor at the edges of their 128 x 128
tiles, with operands that can go straight to LDS and with rows that cannot."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

EPS = {torch.float64: 2.0 ** -53, torch.float32: 2.0 ** -24}


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
# orders whose first panels are followed by trailing updates: whole tiles, one row
# more, one row less; pad 0 or 1 makes the rows aligned or not
@pytest.mark.parametrize("n", [5120, 5121, 5247])
@pytest.mark.parametrize("pad", [0, 1])
def test_trailing_update_edges(n, pad, dtype):
    import linfa_linalg_hip as llh
    g = torch.Generator(device="cuda").manual_seed(n)
    b = torch.randn(n, n, dtype=torch.float64, device="cuda", generator=g)
    a = (b @ b.T / n + torch.eye(n, dtype=torch.float64, device="cuda")).to(dtype)
    w = torch.full((n, n + pad), 9.0, dtype=dtype, device="cuda")
    w[:, :n] = torch.tril(a) + 9.0 * torch.triu(torch.ones_like(a), 1)
    llh.device.potrf(w[:, :n])
    # the strict upper triangle and the padding are untouched
    assert (torch.triu(w[:, :n], 1) == 9.0 * torch.triu(torch.ones_like(a), 1)).all() and (w[:, n:] == 9.0).all()
    l = torch.tril(w[:, :n]).double()
    full = torch.tril(a.double()) + torch.tril(a.double(), -1).T
    err = (full - l @ l.T).norm() / full.norm()
    assert err <= (n + 1) * EPS[dtype] / 16, float(err)  # random signs: far below the bound gamma_n


def test_allocation_free_solve_same_bits_large():
    """The allocation-free solve runs the same updates, to the bit, with rows that
    can and cannot go straight to LDS."""
    import linfa_linalg_hip as llh
    from linfa_linalg_hip import _abi
    import ctypes
    for n, pad in ((4500, 0), (4500, 1)):
        g = torch.Generator(device="cuda").manual_seed(n)
        b = torch.randn(n, n, dtype=torch.float64, device="cuda", generator=g)
        a = b @ b.T / n + torch.eye(n, dtype=torch.float64, device="cuda")
        x = torch.randn(n, 3, dtype=torch.float64, device="cuda", generator=g)
        outs = []
        for form in ("solvec", "solvec_noalloc"):
            w = torch.zeros(n, n + pad, dtype=torch.float64, device="cuda")
            w[:, :n] = a
            y = x.clone()
            c = llh.device.context()
            err = _abi.LlhError()
            st = getattr(c._lib, f"llh_dev_{form}_d")(c.handle, n, ctypes.c_void_p(w.data_ptr()), n + pad, 3,
                                                      ctypes.c_void_p(y.data_ptr()), 3, ctypes.byref(err))
            assert st == 0
            outs.append((w, y))
        assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
