"""The binary64 GEMV whose split of op(A) is fused into the slice products, at the edges of its row
instances (512, 2048 and 8192 elements a row), with more rows than workgroups, beyond its slice counts (8 of
A, 4 of x) and on non-finite data: bitwise the oracle's result and counts."""
import numpy as np
import pytest

from gpu_util import bits_equal, dev, first_diff, host, say, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    torch_cuda()
    import ozblas_amd
    return ozblas_amd


def _run(oz, oracle, m, n, A, x, lda, trans, sumMode):
    ly = m if trans == "N" else n
    y0 = np.linspace(-1.0, 1.0, ly)
    h = oracle.Handle(1 << 30, sumMode=sumMode)
    want = y0.copy()
    h.gemv(trans, m, n, 0.75, A, lda, x, -0.5, want)
    H = oz.Handle(1 << 29, sumMode=sumMode)
    dy = dev(y0)
    say(f"dgemv split {m}x{n} lda={lda} {trans} sumMode={sumMode}")
    H.dgemv(trans, m, n, 0.75, dev(A), lda, dev(x), -0.5, dy)
    assert (H.nSplitA, H.nSplitB) == (h.nSplitA, h.nSplitB)
    return host(dy), want


@pytest.mark.parametrize("k,rows", [(1, 3), (255, 2049), (511, 17), (512, 16), (513, 1030), (2047, 3), (2048, 1025),
                                    (2049, 258), (4096, 257), (8191, 15), (8192, 5), (8193, 5)])
@pytest.mark.parametrize("trans,sumMode,pad", [("T", 1, 1), ("T", 0, 0), ("N", 1, 0)])
def test_row_lengths(oz, oracle, k, rows, trans, sumMode, pad):
    rng = np.random.default_rng(k + rows)
    m, n = (k, rows) if trans == "T" else (rows, k)
    lda = m + pad
    A = rng.standard_normal(lda * n) * np.exp2(rng.integers(-3, 4, lda * n).astype(float))
    got, want = _run(oz, oracle, m, n, A, rng.standard_normal(k), lda, trans, sumMode)
    assert bits_equal(got, want), first_diff(got, want)


@pytest.mark.parametrize("spanA,spanX", [(200, 2), (20, 150), (120, 60), (300, 300)])
@pytest.mark.parametrize("sumMode", [0, 1])
def test_more_slices_than_the_kernel_holds(oz, oracle, spanA, spanX, sumMode):
    rng = np.random.default_rng(spanA)
    m, n = 700, 30
    A = rng.standard_normal(m * n) * np.exp2(rng.integers(-spanA, spanA, m * n).astype(float))
    x = rng.standard_normal(m) * np.exp2(rng.integers(-spanX, spanX, m).astype(float))
    got, want = _run(oz, oracle, m, n, A, x, m, "T", sumMode)
    assert bits_equal(got, want), first_diff(got, want)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("where", ["A", "x"])
def test_non_finite(oz, oracle, bad, where):
    """Non-finite where the oracle's result is; the other rows as the oracle's."""
    rng = np.random.default_rng(7)
    m, n = 600, 20
    A, x = rng.standard_normal(m * n), rng.standard_normal(m)
    (A if where == "A" else x)[5 * m + 77 if where == "A" else 77] = bad
    got, want = _run(oz, oracle, m, n, A, x, m, "T", 1)
    assert np.array_equal(np.isfinite(got), np.isfinite(want))
    assert bits_equal(got[np.isfinite(want)], want[np.isfinite(want)])
