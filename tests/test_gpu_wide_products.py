"""Products of more columns than 65536 workgroups of a launch's second dimension cover: the narrow slices' ordered sum
(4 columns a workgroup), and the residue writers (16), by the plain form with NearSum."""
import numpy as np
import pytest

from gpu_util import bits_equal, dev, first_diff, host, say, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    torch_cuda()
    import ozblas_amd
    return ozblas_amd


@pytest.mark.parametrize("prec,mode", [("s", 0), ("s", 1), ("ds", 0)])
def test_narrow_sum_columns(oz, oracle, prec, mode):
    m, n, k = 3, 262_200, 5
    init = oracle.s_init_mat if prec == "s" else oracle.init_mat
    A, B, C0 = init(m, k, m, 1.0, 2, 1), init(k, n, k, 1.0, 2, 2), init(m, n, m, 1.0, 2, 3)
    one = np.float32 if prec == "s" else float
    want = C0.copy()
    h = oracle.Handle(1 << 32, sumMode=mode)
    getattr(h, prec + "gemm")("n", "n", m, n, k, one(1.25), A, m, B, k, one(-0.5), want, m)
    H = oz.Handle(8 << 30, sumMode=mode)
    C = dev(C0)
    say(f"wide {prec}gemm sumMode={mode}")
    getattr(H, prec + "gemm")("n", "n", m, n, k, 1.25, dev(A), m, dev(B), k, -0.5, C, m)
    assert bits_equal(host(C), want), first_diff(host(C), want)


@pytest.mark.parametrize("m,n", [(2, 1_048_600), (1_048_600, 2)])
def test_residue_writer_columns(oz, oracle, m, n):
    k = 13
    A, B = oracle.init_mat(k, m, k, 0.5, 2, 4), oracle.init_mat(k, n, k, 0.5, 2, 5)
    want = np.zeros(m * n)
    oracle.Handle(1 << 33, sumMode=1).gemm("T", "N", m, n, k, 1.0, A, k, B, k, 0.0, want, m)
    H = oz.Handle(24 << 30, sumMode=1)
    C = dev(np.zeros(m * n))
    say(f"wide residues {m}x{n}x{k}")
    H.dgemm("T", "N", m, n, k, 1.0, dev(A), k, dev(B), k, 0.0, C, m)
    assert (H.mbk, H.nbk) == (m, n)
    assert bits_equal(host(C), want), first_diff(host(C), want)
