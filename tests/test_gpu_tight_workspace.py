"""Products at the smallest workspaces they accept.  The plain NearSum DGEMM: room for the pass that counts the slices, from
none to spare up to the statistics of the residue form beside it.  The product runs in blocks there, bitwise the
oracle's result."""
import numpy as np
import pytest

from gpu_util import bits_equal, dev, first_diff, host, say, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    torch_cuda()
    import ozblas_amd
    return ozblas_amd


@pytest.mark.parametrize("m,n,k", [(600, 590, 256), (20000, 100, 16)])
@pytest.mark.parametrize("spare", [0, 256, 3000, 9000, 100000])
def test_count_pass_just_fits(oz, oracle, m, n, k, spare):
    A, B = oracle.init_mat(k, m, k, 1.0, 2, 1), oracle.init_mat(k, n, k, 1.0, 2, 2)
    want = np.zeros(m * n)
    oracle.Handle(1 << 31, sumMode=1).gemm("T", "N", m, n, k, 1.0, A, k, B, k, 0.0, want, m)
    # the count pass holds a remainder and a slice of the wider operand and a level a column
    work = 16 * k * max(m, n) + 4 * max(m, n) + 512 + spare
    assert work > 1 << 20
    H = oz.Handle(work, sumMode=1)
    C = dev(np.zeros(m * n))
    say(f"tight workspace {m}x{n}x{k} spare={spare}")
    H.dgemm("T", "N", m, n, k, 1.0, dev(A), k, dev(B), k, 0.0, C, m)
    assert bits_equal(host(C), want), first_diff(host(C), want)


@pytest.mark.parametrize("spare", [0, 256])
def test_digit_form_exactly_fits(oz, oracle, spare):
    """Radix-256 digits of small integers (one digit a side, one pair, one 256 x 256 tile shape): the planes, the
    exponents, the tables and the int32 product, and nothing for statistics."""
    m, n, k = 512, 520, 300
    rng = np.random.default_rng(1)
    A, B = rng.integers(-100, 101, m * k).astype(float), rng.integers(-100, 101, n * k).astype(float)

    def up(x, to=256):
        return (x + to - 1) // to * to

    parts = [8 * m, up(k, 128) * up(m), 8 * n, up(k, 128) * up(n), 8, 20, 4, 4, 4 * up(m) * up(n), 128]
    work = sum(map(up, parts)) + 8 * up(m) // 256 * up(n) // 256 + 512 + spare
    assert work > 1 << 20
    want = oracle.exact_gemm_rn("T", "N", m, n, k, A, k, B, k).ravel(order="F")
    H = oz.Handle(work, sumMode=1, sliceType="int8", digitScheme=1)
    C = dev(np.zeros(m * n))
    say(f"tight digits spare={spare}")
    H.dgemm("T", "N", m, n, k, 1.0, dev(A), k, dev(B), k, 0.0, C, m)
    assert (H.schemeUsed, H.nSplitA, H.nSplitB) == (1, 1, 1)
    assert bits_equal(host(C), want), first_diff(host(C), want)
