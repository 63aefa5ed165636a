"""DGEMV of a matrix in which one row alone takes more slices than the fused kernel holds (8): the workgroups stop
early and the stored slices are taken.  Every row instance, the row in a workgroup's first and last share, and split
limits on both sides of 8: bitwise the oracle's result and counts."""
import numpy as np
import pytest

from gpu_util import bits_equal, dev, first_diff, host, say, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    torch_cuda()
    import ozblas_amd
    return ozblas_amd


@pytest.mark.parametrize("k,rows", [(300, 5000), (2000, 2300), (4000, 700)])
@pytest.mark.parametrize("where", [0, 0.5, 1])
@pytest.mark.parametrize("flags", [dict(sumMode=1), dict(sumMode=0, nSplitMax=8), dict(sumMode=1, nSplitMax=9)],
                         ids=lambda f: ",".join(f"{a}={b}" for a, b in f.items()))
def test_one_long_row(oz, oracle, k, rows, where, flags):
    rng = np.random.default_rng(rows)
    A = rng.standard_normal((rows, k))
    r = int(where * (rows - 1))
    A[r] *= np.exp2(rng.integers(-150, 150, k).astype(float))
    A = A.ravel()
    x, y0 = rng.standard_normal(k), np.linspace(-1.0, 1.0, rows)
    h = oracle.Handle(1 << 31, **flags)
    want = y0.copy()
    h.gemv("T", k, rows, 0.75, A, k, x, -0.5, want)
    H = oz.Handle(1 << 30, **flags)
    dy = dev(y0)
    say(f"dgemv one long row {k}x{rows} row={r} {flags}")
    for _ in range(2):
        dy = dev(y0)
        H.dgemv("T", k, rows, 0.75, dev(A), k, dev(x), -0.5, dy)
        assert bits_equal(host(dy), want), first_diff(host(dy), want)
        assert (H.nSplitA, H.nSplitB) == (h.nSplitA, h.nSplitB)
