"""FP16 and BF16 residue planes, which are taken where the INT8 planes (padded to 256 columns) do not fit: workspaces
between the two needs, with several product tiles of odd edges, sums past one binary32 flush (k > 1024), two k chunks
(k > 65536), wide spans and cancellation.  Every element the exact product rounded once."""
import numpy as np
import pytest

from gpu_util import bits_equal, dev, first_diff, host, say, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    torch_cuda()
    import ozblas_amd
    return ozblas_amd


def _up(x, to):
    return (x + to - 1) // to * to


def _needs(m, n, k, nmod):
    """Bytes of the planes and product residues, half and INT8 (transposed operands: no copies)."""
    half = 2 * _up(k, 64) * (m + n) + _up(m, 64) * _up(n, 4) * ((_up(k, 64) + 65535) // 65536)
    int8 = _up(k, 128) * (_up(m, 256) + _up(n, 256)) + _up(m, 256) * _up(n, 256) * ((_up(k, 128) + 65535) // 65536)
    return half * nmod, int8 * nmod


@pytest.mark.parametrize("form", ["fp16", "bf16"])
@pytest.mark.parametrize("m,n,k", [(3, 5, 1), (129, 130, 63), (131, 129, 1100), (130, 70, 2049), (33, 200, 4097),
                                   (130, 3, 66000), (5, 3, 131200)])
@pytest.mark.parametrize("kind", ["full", "span", "cancel"])
def test_half_planes(oz, oracle, form, m, n, k, kind):
    rng = np.random.default_rng(m + n + k)
    A, B = rng.standard_normal((m, k)), rng.standard_normal((n, k))
    if kind == "span":
        A *= np.exp2(rng.integers(-30, 31, (m, k)).astype(float))
        B *= np.exp2(rng.integers(-6, 7, (n, k)).astype(float))
    elif kind == "cancel" and k > 1:  # the second half of the sum takes back the first but for a few last bits
        h = k // 2
        A[:, h:2 * h], B[:, h:2 * h] = -A[:, :h], B[:, :h]
        A[:, h] *= 1 + 2.0 ** -40
    A, B = A.ravel(), B.ravel()
    want = oracle.exact_gemm_rn("T", "N", m, n, k, A, k, B, k).ravel(order="F")
    dA, dB = dev(A), dev(B)

    def run(work):
        H = oz.Handle(work, sumMode=1, sliceType=form, digitScheme=2)
        C = dev(np.zeros(m * n))
        say(f"half planes {form} {m}x{n}x{k} {kind} work={work}")
        H.dgemm("T", "N", m, n, k, 1.0, dA, k, dB, k, 0.0, C, m)
        assert H.schemeUsed == 2
        assert bits_equal(host(C), want), first_diff(host(C), want)
        return int(H.nSplitC)

    nmod = run(4 << 30)
    half, int8 = _needs(m, n, k, nmod)
    work = max(half + 200_000, 1 << 20)  # statistics, items and alignment beside the planes
    assert work < int8, "the INT8 planes would fit"
    assert run(work) == nmod
