"""The residue form's reconstruction at every word count of its kernels and at the edges of its 32 x 4
wave tiles, against the exact product in Python integers (rounded once by float()): few to many moduli
(the matrix-unit kernels of 4, 6 and 8 words up to 32 moduli, the scalar one beyond), rows and columns
around 32 and 4, zeros, exact cancellation and alpha / beta."""
import random
from fractions import Fraction as Fr

import numpy as np
import pytest

from gpu_util import bits_equal, dev, first_diff, host, say, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    torch_cuda()
    import ozblas_amd
    return ozblas_amd


# element bits and largest shift: about (2 (bits + shift) + log2 k + 2) / 7.9 moduli
@pytest.mark.parametrize("bits,shift", [(1, 0), (4, 2), (12, 0), (30, 0), (53, 0), (53, 18), (53, 34), (53, 50), (53, 64),
                                        (53, 90)])
@pytest.mark.parametrize("m,n,k", [(1, 1, 3), (31, 3, 17), (32, 4, 16), (33, 5, 40), (70, 9, 8), (129, 1, 5)])
def test_residue_reconstruction_exact(oz, m, n, k, bits, shift):
    rng = random.Random(bits * 1000 + shift * 10 + m)
    val = lambda: (1 if rng.random() < 0.5 else -1) * (rng.getrandbits(bits) | 1) << rng.randint(0, shift)
    A = [[val() if rng.random() < 0.9 else 0 for _ in range(k)] for _ in range(m)]
    B = [[val() if rng.random() < 0.9 else 0 for _ in range(n)] for _ in range(k)]
    if k > 2:  # row 0 times column 0 cancels exactly
        A[0][0], A[0][1], B[0][0], B[1][0] = 3, -3, 5, 5
        for q in range(2, k):
            A[0][q] = 0
    X = [[sum(A[i][q] * B[q][j] for q in range(k)) for j in range(n)] for i in range(m)]
    flat = lambda W, r, c: np.array([float(W[i][j]) for j in range(c) for i in range(r)])
    C0 = np.array([float(rng.randint(-9, 9)) for _ in range(m * n)])
    want = np.array([float(Fr(2) * Fr(x) + Fr(-0.5) * Fr(c)) for x, c in zip(flat(X, m, n).tolist(), C0.tolist())])
    H = oz.Handle(1 << 28, sumMode=1, sliceType="int8", digitScheme="residues")
    dC = dev(C0)
    say(f"residue recon {m}x{n}x{k} bits={bits} shift={shift}")
    H.dgemm("N", "N", m, n, k, 2.0, dev(flat(A, m, k)), m, dev(flat(B, k, n)), k, -0.5, dC, m)
    assert H.schemeUsed == 2
    assert bits_equal(host(dC), want), first_diff(host(dC), want)


def test_matmul_result_memory_is_not_an_input():
    """beta = 0 multiplies C rather than dropping it (as the reference does), so the product must not start from
    recycled memory: NaN left in it came out in the result."""
    torch = torch_cuda()
    from ozblas_amd.autograd import ozaki_mm
    A, B = torch.ones((7, 5), dtype=torch.float64).cuda(), torch.ones((5, 6), dtype=torch.float64).cuda()
    for form in ("int8", "fp16"):
        for _ in range(3):
            left = torch.full((7, 6), float("nan"), dtype=torch.float64, device="cuda")
            del left  # back to the allocator, which hands it out for the next 7 x 6
            assert bool((ozaki_mm(A, B, form) == 5.0).all())
