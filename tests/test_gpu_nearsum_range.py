"""NearSum of finite terms so near overflow that the unit of its first transform is not finite.  The reference's loop does
not end there; every routine here returns, with NaN, and its next call is as ever."""
import numpy as np
import pytest

from gpu_util import dev, host, say, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    torch_cuda()
    import ozblas_amd
    return ozblas_amd


def _near_top(single, n, k):
    """A matrix and a vector whose products are finite and within a factor 4 of overflow."""
    top = (64, 62) if single else (512, 510)
    dtype = np.float32 if single else np.float64
    rng = np.random.default_rng(n + k)
    A = ((1 + rng.random(n * k)) * 2.0 ** (top[0] - 1)).astype(dtype)
    x = np.zeros(k, dtype)
    x[0] = 1.75 * 2.0 ** top[1]
    return A, x


@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("n", [1, 300, 20_000])
def test_dot(oz, single, n):
    A, x = _near_top(single, 1, n)
    H = oz.Handle(1 << 28, sumMode=1)
    f = H.sdot if single else H.ddot
    say(f"near top dot single={single} n={n}")
    assert np.isnan(f(n, dev(A), dev(x)))
    one = dev(np.ones(n, A.dtype))
    assert f(n, one, one) == n


@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("m,n,k", [(5, 1, 300), (5, 4, 300), (1, 1, 40)])
def test_gemm(oz, single, m, n, k):
    A, x = _near_top(single, m, k)
    H = oz.Handle(1 << 28, sumMode=1)
    C = dev(np.zeros(m * n, A.dtype))
    B = np.tile(x, n)
    f = H.sgemm if single else H.dgemm
    say(f"near top gemm single={single} {m}x{n}x{k}")
    f("T", "N", m, n, k, 1.0, dev(A), k, dev(B), k, 0.0, C, m)
    assert np.isnan(host(C)).all()
    C = dev(np.zeros(m * n, A.dtype))
    f("T", "N", m, n, k, 1.0, dev(np.ones_like(A)), k, dev(np.ones_like(B)), k, 0.0, C, m)
    assert (host(C) == k).all()


@pytest.mark.parametrize("single", [False, True])
def test_csrmv(oz, single):
    m, k = 300, 3
    A, _ = _near_top(single, m, k)
    rowptr = np.arange(0, m * k + 1, k).astype(np.int32)
    colind = np.tile(np.arange(k), m).astype(np.int32)
    x = np.full(m, A.dtype.type(1.75 * 2.0 ** (61 if single else 509)))
    H = oz.Handle(1 << 28, sumMode=1)
    f = H.scsrmv if single else H.dcsrmv
    y = dev(np.zeros(m, A.dtype))
    say(f"near top csrmv single={single}")
    f(m, m, m * k, 1.0, dev(A), dev(colind), dev(rowptr), dev(x), 0.0, y)
    assert np.isnan(host(y)).all()
    y, one = dev(np.zeros(m, A.dtype)), dev(np.ones(m, A.dtype))
    f(m, m, m * k, 1.0, dev(np.ones_like(A)), dev(colind), dev(rowptr), one, 0.0, y)
    assert (host(y) == k).all()
