"""Binary32 vectors of more than 65536 elements, whose slices hold one to three bits: the sparse product and the CG with
up to 32 slices in registers, slice dots of 17 to 32 slices a side on the FP64 matrix units, and the general paths
behind them (more slices, a remainder slot, plans outside the model).  Bitwise the oracle's results and counts."""
import numpy as np
import pytest

from gpu_util import dev, host, say, torch_cuda
from test_gpu_binary32 import _laplace_f, f32_diff, f32_equal

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    torch_cuda()
    import ozblas_amd
    return ozblas_amd


def _vector(rng, n, spread):
    return (rng.standard_normal(n) * np.exp2(rng.integers(-spread, spread + 1, n).astype(float))).astype(np.float32)


def _matrix(rng, m, n, bits):
    """Rows of 0 to 9 entries, some sums of exactly cancelling pairs, a run of long rows; values of `bits` bits."""
    length = rng.integers(0, 10, m)
    length[m // 2 : m // 2 + 3] = 900
    rowptr = np.concatenate([[0], np.cumsum(length)]).astype(np.int32)
    nnz = int(rowptr[-1])
    colind = rng.integers(0, n, nnz).astype(np.int32)
    val = rng.integers(1 - (1 << bits), 1 << bits, nnz).astype(np.float32) * np.float32(2.0 ** -bits)
    for r in range(0, m, 50):  # a x - a x: no clear-cut sum
        b, e = rowptr[r], rowptr[r + 1]
        if e - b >= 2:
            val[b:e] = 0
            colind[b + 1], val[b], val[b + 1] = colind[b], 0.375, -0.375
    return rowptr, nnz, colind, val


@pytest.mark.parametrize("n,spread", [(65_537, 0), (70_000, 6), (262_145, 2)])
@pytest.mark.parametrize("bits", [6, 23])  # two slices of A, and three or four
@pytest.mark.parametrize("flags", [dict(sumMode=1), dict(sumMode=0), dict(sumMode=1, fastMode=2),
                                   dict(sumMode=1, reproMode=0), dict(sumMode=1, nSplitMax=70)],
                         ids=lambda f: ",".join(f"{a}={b}" for a, b in f.items()))
@pytest.mark.parametrize("presplit", [False, True])
def test_sparse_product(oz, oracle, n, spread, bits, flags, presplit):
    m = 3001
    rng = np.random.default_rng(n + bits)
    rowptr, nnz, colind, val = _matrix(rng, m, n, bits)
    x, y0 = _vector(rng, n, spread), rng.standard_normal(m).astype(np.float32)
    h, H = oracle.Handle(1 << 32, **flags), oz.Handle(1 << 30, **flags)
    want, dy = y0.copy(), dev(y0)
    dval, dcol, drow = dev(val), dev(colind), dev(rowptr)
    say(f"long scsrmv n={n} spread={spread} bits={bits} {flags} presplit={presplit}")
    hA, A = val, dval
    if presplit:
        hA, A = h.scsrmv_splitA(m, n, nnz, val, rowptr), H.scsrmv_splitA(m, n, nnz, dval, drow)
        assert (H.nSplitA_, H.splitShift) == (h.nSplitA_, h.splitShift)
    h.scsrmv(m, n, nnz, np.float32(1.25), hA, colind, rowptr, x, np.float32(-0.5), want)
    H.scsrmv(m, n, nnz, 1.25, A, dcol, drow, dev(x), -0.5, dy)
    assert (H.nSplitA, H.nSplitB) == (h.nSplitA, h.nSplitB)
    assert H.nSplitB > 8
    assert f32_equal(host(dy), want), f32_diff(host(dy), want)


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_sparse_product_non_finite(oz, oracle, bad):
    m = n = 66_000
    rng = np.random.default_rng(1)
    rowptr, nnz, colind, val = _matrix(rng, m, n, 6)
    x, y0 = _vector(rng, n, 1), np.zeros(m, np.float32)
    x[12_345] = bad
    want, dy = y0.copy(), dev(y0)
    oracle.Handle(1 << 32, sumMode=1).scsrmv(m, n, nnz, np.float32(1), val, colind, rowptr, x, np.float32(0), want)
    say(f"long scsrmv bad={bad}")
    oz.Handle(1 << 30, sumMode=1).scsrmv(m, n, nnz, 1.0, dev(val), dev(colind), dev(rowptr), dev(x), 0.0, dy)
    got, ok = host(dy), np.isfinite(want)
    assert not ok.all() and np.array_equal(np.isfinite(got), ok)
    assert f32_equal(got[ok], want[ok]), f32_diff(got[ok], want[ok])


@pytest.mark.parametrize("flags", [dict(sumMode=1), dict(sumMode=0), dict(sumMode=1, nSplitMax=70),
                                   dict(sumMode=1, cgDeviceSlices=9)],
                         ids=lambda f: ",".join(f"{a}={b}" for a, b in f.items()))
def test_cg(oz, oracle, flags):
    g, iters = 41, 5
    rowptr, colind, val, n, nnz = _laplace_f(oracle, g)
    assert n > 65536
    b = np.random.default_rng(g).uniform(-1, 1, n).astype(np.float32)
    ref = {k: v for k, v in flags.items() if k != "cgDeviceSlices"}
    xw, dx = np.zeros(n, dtype=np.float32), dev(np.zeros(n, dtype=np.float32))
    want = oracle.Handle(1 << 32, **ref).scg(n, nnz, val, colind, rowptr, b, xw, iters, np.float32(0))
    H = oz.Handle(1 << 30, **flags)
    say(f"long scg n={n} {flags}")
    got = H.scg(n, nnz, dev(val), dev(colind), dev(rowptr), dev(b), dx, iters, 0.0)
    # a vector of more than 9 slices takes the solve to the synchronous path
    assert H.cgDevicePath == (2 if "cgDeviceSlices" in flags else 1)
    assert f32_equal(got.astype(np.float32), want), f32_diff(got, want)
    assert f32_equal(host(dx), xw), f32_diff(host(dx), xw)


@pytest.mark.parametrize("n,spreads", [(70_000, (18, 18)), (70_001, (1, 30)), (1_000_003, (8, 4)), (300_000, (16, 30))])
@pytest.mark.parametrize("flags", [dict(sumMode=1), dict(sumMode=0), dict(sumMode=1, reproMode=0),
                                   dict(sumMode=1, nSplitMax=40)],
                         ids=lambda f: ",".join(f"{a}={b}" for a, b in f.items()))
def test_dot(oz, oracle, n, spreads, flags):
    rng = np.random.default_rng(n)
    x, y = _vector(rng, n, spreads[0]), _vector(rng, n, spreads[1])
    h, H = oracle.Handle(1 << 34, **flags), oz.Handle(1 << 32, **flags)
    dx, dy = dev(x), dev(y)
    say(f"long sdot n={n} {spreads} {flags}")
    want = np.float32(h.sdot(n, x, y))
    for _ in range(2):  # the second call meets the scratch the first one left
        got = np.float32(H.sdot(n, dx, dy))
        assert (H.nSplitA, H.nSplitB) == (h.nSplitA, h.nSplitB)
        assert max(H.nSplitA, H.nSplitB) > 16
        assert got.view(np.uint32) == want.view(np.uint32)
    want = np.float32(oracle.Handle(1 << 34, **flags).snrm2(n, x))
    assert np.float32(H.snrm2(n, dx)).view(np.uint32) == want.view(np.uint32)
