"""Which products the plain NearSum DGEMM ran, told by the operations it reports (2 m n k for each slice pair, or for
each modulus): both sides of the lines between FP64 slices and residues, the calls that keep the slices, and an operand
of zeros, which needs no products.  Bitwise the oracle's result on either path."""
import numpy as np
import pytest

from gpu_util import bits_equal, dev, first_diff, host, say, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    torch_cuda()
    import ozblas_amd
    return ozblas_amd


def _run(oz, oracle, m, n, k, A, B, **flags):
    flags = {"sumMode": 1, **flags}
    want = np.zeros(m * n)
    h = oracle.Handle(1 << 31, **flags)
    h.gemm("T", "N", m, n, k, 1.0, A, k, B, k, 0.0, want, m)
    H = oz.Handle(1 << 31, **flags)
    C = dev(np.zeros(m * n))
    say(f"plain path {m}x{n}x{k} {flags}")
    H.dgemm("T", "N", m, n, k, 1.0, dev(A), k, dev(B), k, 0.0, C, m)
    assert bits_equal(host(C), want), first_diff(host(C), want)
    assert (H.nSplitA, H.nSplitB, H.schemeUsed) == (h.nSplitA, h.nSplitB, 0)
    return H, round(H.n_comp / (2.0 * m * n * k), 3)


@pytest.mark.parametrize("m,n,k,taken", [
    (1000, 195, 128, False),   # 2.496e7 multiply-adds, below 2.5e7
    (1000, 196, 128, True),    # 2.509e7
    (40, 41, 255, False),
    (40, 41, 256, True),
    (2, 2, 8191, True),
])
def test_both_sides_of_the_line(oz, oracle, m, n, k, taken):
    rng = np.random.default_rng(k)
    # full mantissas over a few binades: four slices a side
    A, B = (rng.standard_normal(s * k) * np.exp2(rng.integers(-8, 9, s * k).astype(float)) for s in (m, n))
    H, products = _run(oz, oracle, m, n, k, A, B)
    assert (H.nSplitA, H.nSplitB) == (4, 4)
    assert (products != 16) == taken
    if taken:
        assert products == int(products) and 17 <= products <= 30


@pytest.mark.parametrize("flags", [dict(fastMode=1), dict(nSplitMax=4), dict(sumMode=0)], ids=str)
def test_slices_kept(oz, oracle, flags):
    """Dropped slices and the ordered sum."""
    rng = np.random.default_rng(3)
    m, n, k = 90, 80, 300
    H, products = _run(oz, oracle, m, n, k, rng.standard_normal(m * k), rng.standard_normal(n * k), **flags)
    assert products == H.nSplitC


@pytest.mark.parametrize("m,n,k", [(2, 2, 256), (90, 80, 300), (1000, 196, 128)])
def test_few_slices(oz, oracle, m, n, k):
    """Small integers, two slices a side: with the statistics there, the few moduli that cover them."""
    rng = np.random.default_rng(3)
    A, B = (rng.integers(-7, 8, s * k).astype(float) for s in (m, n))
    H, products = _run(oz, oracle, m, n, k, A, B)
    assert H.nSplitA * H.nSplitB == 4 and products < 4


@pytest.mark.parametrize("form", ["fp64", "int8"])
def test_zero_operand_reports_no_products(oz, form):
    m, n, k = 64, 60, 400
    rng = np.random.default_rng(4)
    H = oz.Handle(1 << 28, sumMode=1, sliceType=form)
    B, C = dev(rng.standard_normal(n * k)), dev(np.full(m * n, 7.0))
    H.dgemm("T", "N", m, n, k, 1.0, dev(rng.standard_normal(m * k)), k, B, k, 0.0, C, m)
    assert H.n_comp > 0
    say(f"zero operand {form}")
    H.dgemm("T", "N", m, n, k, 1.0, dev(np.zeros(m * k)), k, B, k, 0.5, C, m)
    assert (H.t_comp, H.t_sum, H.n_comp) == (0.0, 0.0, 0.0)
