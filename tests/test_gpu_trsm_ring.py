"""The blocks that a one-launch triangular solve hands on through its ring of slots:
fewer and more block rows than slots, ragged ends, more column chunks than a launch
has rings for, and solves that follow each other in the same memory."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

EPS = {torch.float64: 2.0 ** -53, torch.float32: 2.0 ** -24}


def _check(n, m, dtype, upper, trans, seed):
    import linfa_linalg_hip as llh
    g = torch.Generator().manual_seed(seed)
    t = torch.randn(n, n, generator=g, dtype=torch.float64) * (0.5 / n ** 0.5)
    t = torch.triu(t, 1) if upper != trans else torch.tril(t, -1)
    t.diagonal().add_(1.0 + torch.rand(n, generator=g, dtype=torch.float64))
    a = t.to(dtype)
    b = torch.randn(n, m, generator=g, dtype=torch.float64).to(dtype)
    x = b.cuda()
    llh.device.solve_triangular(a.cuda(), x, llh.UPLO.Upper if upper else llh.UPLO.Lower, trans=trans)
    op, x = (a.T if trans else a).double(), x.cpu().double()
    res = torch.linalg.norm(op @ x - b.double())
    # the residual of a substitution, gamma_n || |A| |x| ||, with a factor 4 for the
    # inverses of well-conditioned 64 x 64 blocks
    assert res <= 4 * (n + 64) * EPS[dtype] * torch.linalg.norm(op.abs() @ x.abs())


@pytest.mark.parametrize("upper,trans", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
# 1 to 6 block rows (the ring's readers and the first flag); 8, 9 and 17 (laps); 2049
# columns (more chunks than rings)
@pytest.mark.parametrize("n,m", [(64, 1), (100, 3), (129, 16), (255, 17), (321, 5), (384, 64), (512, 9), (513, 33),
                                 (1050, 2), (130, 2049)])
def test_ring_sizes(n, m, dtype, upper, trans):
    _check(n, m, dtype, upper, trans, n + m)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_solves_in_turn(dtype):
    """Larger and smaller solves in one context: no block of an earlier one is taken."""
    for i, (n, m) in enumerate([(1300, 16), (600, 40), (1300, 16), (200, 16), (700, 100), (1300, 1)]):
        _check(n, m, dtype, i % 2 == 0, i % 3 == 0, i)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_epochs_start_anew(dtype):
    """The solves before and after the context's epochs run out (set from here: the
    member in front of the spin limit, found by a value of that)."""
    import ctypes

    from linfa_linalg_hip import device as dev
    _check(600, 40, dtype, False, False, 1)  # the buffers exist
    h = dev.context().handle
    base = h.value if isinstance(h, ctypes.c_void_p) else int(h)
    mark = 0x5A3C1D97E
    dev.set_solve_spin_limit(mark)
    try:
        at = next(o for o in range(8, 2048, 8) if ctypes.c_int64.from_address(base + o).value == mark)
    finally:
        dev.set_solve_spin_limit(0)
    epoch = ctypes.c_int32.from_address(base + at - 8)
    assert 1 < epoch.value < 1 << 30
    epoch.value = 2 ** 31 - 4
    for i in range(4):
        _check(600, 40, dtype, i % 2 == 1, False, i)  # two epochs each
    assert epoch.value < 100
