"""The narrow-slice GEMM (INT8 / FP16 products of the binary32 and mixed routines, oz_narrow.hip) at
the edges of its rules and tiles, bitwise against the oracle: k around the INT8 / FP16 line (1024) and
at the ends of the FP16 range, both INT8 tile sizes, columns of every thread mapping of the split,
pair groups that do not fit the workspace at once, and products in the subnormal range."""
import numpy as np
import pytest

from gpu_util import bits_equal, dev, first_diff, host, say, torch_cuda
from test_gpu_binary32 import f32_diff, f32_equal

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    torch_cuda()
    import ozblas_amd
    return ozblas_amd


SHAPES = [
    # m, n, k, transA, transB
    (2, 2, 1, "n", "n"),          # 12 bits: the FP64 products
    (5, 3, 2, "n", "n"),          # 11 bits, the widest FP16 slice
    (65, 129, 64, "t", "n"),
    (129, 127, 1024, "n", "t"),   # 7 bits: FP16
    (129, 127, 1025, "n", "t"),   # 6 bits: INT8, 128-wide tiles
    (512, 513, 1040, "t", "n"),   # INT8, 256-wide tiles
    (3, 130, 2100, "n", "n"),     # one workgroup per column in the split
    (4, 5, 4200, "t", "t"),
    (3, 2, 8200, "n", "n"),       # 1024 threads per column
    (2, 3, 33000, "n", "n"),      # past the split kernel's columns: the FP64 products
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda c: "x".join(map(str, c[:3])) + c[3] + c[4])
@pytest.mark.parametrize("kind", ["s0", "s1", "ds"])
def test_narrow_gemm_bitwise(oz, oracle, shape, kind):
    m, n, k, ta, tb = shape
    say(f"narrow gemm {kind} {m}x{n}x{k} {ta}{tb}")
    ra, ca = (m, k) if ta == "n" else (k, m)
    rb, cb = (k, n) if tb == "n" else (n, k)
    s = kind[0] == "s"
    mat = (lambda r, c, sd: oracle.s_init_mat(r, c, r, 1.0, 2, sd)) if s else \
        (lambda r, c, sd: oracle.init_mat(r, c, r, 1.0, 2, sd))
    A, B, C0 = mat(ra, ca, 1), mat(rb, cb, 2), mat(m, n, 3)
    A[: ra if ta == "t" else 1] = 0  # a zero column of the stored A, or one zero element
    mode = 1 if kind == "s1" else 0
    want = C0.copy()
    h = oracle.Handle(1 << 32, sumMode=mode)
    one = np.float32 if s else float
    getattr(h, "sgemm" if s else "dsgemm")(ta, tb, m, n, k, one(1.25), A, ra, B, rb, one(-0.5), want, m)
    H = oz.Handle(1 << 30, sumMode=mode)
    dC = dev(C0)
    getattr(H, "sgemm" if s else "dsgemm")(ta, tb, m, n, k, 1.25, dev(A), ra, dev(B), rb, -0.5, dC, m)
    got = host(dC)
    assert (f32_equal(got, want), f32_diff(got, want)) == (True, None) if s else \
        (bits_equal(got, want), first_diff(got, want)) == (True, None)
    assert (H.nSplitA, H.nSplitB, H.nSplitC) == (h.nSplitA, h.nSplitB, h.nSplitC)


@pytest.mark.parametrize("flags", [dict(), dict(fastMode=1), dict(nSplitMax=3), dict(reproMode=0)],
                         ids=lambda f: ",".join(f"{k}={v}" for k, v in f.items()) or "default")
def test_narrow_pair_groups_bitwise(oz, oracle, flags):
    """A workspace that holds the slices but not every pair's product plane: the sum carries over."""
    m, n, k = 200, 190, 1100
    A, B = oracle.s_init_mat(m, k, m, 1.0, 2, 4), oracle.s_init_mat(k, n, k, 1.0, 2, 5)
    want = np.zeros(m * n, dtype=np.float32)
    oracle.Handle(1 << 30, **flags).sgemm("n", "n", m, n, k, np.float32(1), A, m, B, k, np.float32(0), want, m)
    H = oz.Handle(24 << 20, **flags)
    dC = dev(np.zeros(m * n, dtype=np.float32))
    say(f"narrow groups {flags}")
    H.sgemm("n", "n", m, n, k, 1.0, dev(A), m, dev(B), k, 0.0, dC, m)
    assert (H.mbk, H.nbk) == (m, n)
    assert f32_equal(host(dC), want), f32_diff(host(dC), want)


@pytest.mark.parametrize("k", [300, 1100])
def test_narrow_subnormal_products_bitwise(oz, oracle, k):
    m, n = 40, 33
    A, B = oracle.s_init_mat(m, k, m, 2.0, 2, 6), oracle.s_init_mat(k, n, k, 2.0, 2, 7)
    A, B = A * np.float32(2.0 ** -75), B * np.float32(2.0 ** -70)
    want = np.zeros(m * n, dtype=np.float32)
    oracle.Handle(1 << 30).sgemm("n", "n", m, n, k, np.float32(1), A, m, B, k, np.float32(0), want, m)
    H = oz.Handle(1 << 28)
    dC = dev(np.zeros(m * n, dtype=np.float32))
    say(f"narrow subnormal k={k}")
    H.sgemm("n", "n", m, n, k, 1.0, dev(A), m, dev(B), k, 0.0, dC, m)
    assert f32_equal(host(dC), want), f32_diff(host(dC), want)
