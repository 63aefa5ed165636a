"""The plain form with NearSum computed by residues (large products with a complete split): bitwise the oracle's
result and slice counts over transpositions, pads, alpha and beta, on both sides of the line from which it is taken,
and where it must not be taken (dropped slices, other units, ends of the exponent range, non-finite data, a
workspace that does not hold the residue planes)."""
import numpy as np
import pytest

from gpu_util import bits_equal, dev, first_diff, host, say, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    torch_cuda()
    import ozblas_amd
    return ozblas_amd


def _run(oz, oracle, m, n, k, ta="N", tb="N", pad=0, alpha=1.0, beta=0.0, expA=3, expB=3, work=1 << 30, scale=1.0,
         bad=None, zeros=False, **flags):
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    ra, ca = (m, k) if ta == "N" else (k, m)
    rb, cb = (k, n) if tb == "N" else (n, k)
    A = rng.standard_normal((ra + pad) * ca) * np.exp2(rng.integers(-expA, expA + 1, (ra + pad) * ca).astype(float))
    B = rng.standard_normal((rb + pad) * cb) * np.exp2(rng.integers(-expB, expB + 1, (rb + pad) * cb).astype(float))
    A *= scale
    if zeros:
        A[:] = 0.0
    if bad is not None:
        A[11] = bad
    C0 = np.linspace(-1, 1, (m + pad) * n)
    flags = {"sumMode": 1, **flags}
    h = oracle.Handle(1 << 31, **flags)
    want = C0.copy()
    h.gemm(ta, tb, m, n, k, alpha, A, ra + pad, B, rb + pad, beta, want, m + pad)
    H = oz.Handle(work, **flags)
    C = dev(C0)
    say(f"plain residue {m}x{n}x{k} {ta}{tb} pad={pad} {flags} scale={scale} bad={bad}")
    H.dgemm(ta, tb, m, n, k, alpha, dev(A), ra + pad, dev(B), rb + pad, beta, C, m + pad)
    return host(C), want, H, h


@pytest.mark.parametrize("m,n,k,kw", [
    (300, 290, 700, {}),
    (300, 290, 700, dict(ta="T", tb="N", pad=1, alpha=0.75, beta=-0.5)),
    (300, 290, 700, dict(ta="N", tb="T", pad=3, alpha=-1.0, beta=1.0)),
    (300, 290, 700, dict(ta="T", tb="T", reproMode=0)),
    (2, 2, 8191, {}),                      # below the line
    (17, 600, 6000, dict(beta=2.0)),
    (1000, 2, 20000, dict(ta="T")),        # beyond the register split
    (257, 400, 513, dict(expA=60, expB=2)),
    (257, 400, 513, dict(expA=100, expB=100)),
    (400, 400, 400, dict(zeros=True, beta=0.5)),
    (400, 400, 400, dict(scale=2.0 ** 880)),
], ids=str)
def test_same_bits_and_counts(oz, oracle, m, n, k, kw):
    got, want, H, h = _run(oz, oracle, m, n, k, **kw)
    assert (H.nSplitA, H.nSplitB) == (h.nSplitA, h.nSplitB)
    assert H.schemeUsed == 0
    assert bits_equal(got, want), first_diff(got, want)


@pytest.mark.parametrize("kw", [dict(nSplitMax=2), dict(nSplitMax=12), dict(fastMode=1),
                                dict(scale=2.0 ** -1000, expA=1), dict(scale=2.0 ** 960, expB=1), dict(work=40 << 20)],
                         ids=str)
def test_not_taken(oz, oracle, kw):
    """The FP64 products' own results: rounded or dropped terms, scaled data; and a tight workspace."""
    got, want, H, h = _run(oz, oracle, 300, 290, 700, **kw)
    assert bits_equal(got, want), first_diff(got, want)


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_non_finite(oz, oracle, bad):
    got, want, _, _ = _run(oz, oracle, 300, 290, 700, bad=bad)
    assert np.array_equal(np.isfinite(got), np.isfinite(want))
    ok = np.isfinite(want)
    assert bits_equal(got[ok], want[ok])


@pytest.mark.parametrize("form", ["fp16", "bf16"])
@pytest.mark.parametrize("m,n,k", [(3, 5, 700), (70, 33, 129), (130, 260, 500)])
@pytest.mark.parametrize("work", [1 << 30, 4 << 20])
def test_half_forms_residues(oz, oracle, form, m, n, k, work):
    """FP16 and BF16 residues: INT8 planes, or planes of their own where a tight workspace does not hold those."""
    rng = np.random.default_rng(m)
    A, B = rng.standard_normal(m * k), rng.standard_normal(k * n)
    want = oracle.exact_gemm_rn("N", "N", m, n, k, A, m, B, k).ravel(order="F")  # m x n to column-major
    H = oz.Handle(work, sumMode=1, sliceType=form, digitScheme=2)
    C = dev(np.zeros(m * n))
    say(f"half form {form} {m}x{n}x{k} work={work}")
    try:
        H.dgemm("N", "N", m, n, k, 1.0, dev(A), m, dev(B), k, 0.0, C, m)
    except Exception as e:  # 130 x 260 x 500 needs more than 4 MB in either layout
        assert work == 4 << 20 and m == 130, e
        return
    assert H.schemeUsed == 2
    assert bits_equal(host(C), want), first_diff(host(C), want)
