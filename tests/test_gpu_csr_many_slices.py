"""Sparse products whose vector takes more slices than the staged kernel's registers hold: its slices are stored from
the plan already made, or were stored with it where the plan is outside the model (a split limit beyond the plan's
levels, a non-finite element).  Bitwise the oracle's result and counts."""
import numpy as np
import pytest

from gpu_util import bits_equal, dev, first_diff, host, say, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    torch_cuda()
    import ozblas_amd
    return ozblas_amd


def _problem(n, m, seed, single):
    rng = np.random.default_rng(seed)
    length = rng.integers(0, 12, m)
    rowptr = np.concatenate([[0], np.cumsum(length)]).astype(np.int32)
    nnz = int(rowptr[-1])
    colind = rng.integers(0, n, nnz).astype(np.int32)
    spread = 40 if single else 150
    x = rng.standard_normal(n) * np.exp2(rng.integers(-spread, spread, n).astype(float))
    dtype = np.float32 if single else np.float64
    return rowptr, nnz, colind, rng.standard_normal(nnz).astype(dtype), x.astype(dtype)


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("m,n", [(1, 300), (300, 300), (20, 5000), (3000, 40)])
@pytest.mark.parametrize("flags", [dict(sumMode=1), dict(sumMode=0), dict(sumMode=1, reproMode=0),
                                   dict(sumMode=1, nSplitMax=70), dict(sumMode=1, nSplitMax=9)],
                         ids=lambda f: ",".join(f"{a}={b}" for a, b in f.items()))
@pytest.mark.parametrize("bad", [None, np.inf])
def test_vector_of_many_slices(oz, oracle, prec, m, n, flags, bad):
    if bad is not None and flags.get("reproMode") == 0:
        pytest.skip("which rows are non-finite with a remainder slot beside an infinity is not pinned")
    single = prec == "s"
    rowptr, nnz, colind, val, x = _problem(n, m, 3 * m + n, single)
    if bad is not None:
        x[n // 2] = bad
    y0 = np.linspace(-1, 1, m).astype(val.dtype)
    one = np.float32 if single else float
    h, H = oracle.Handle(1 << 30, **flags), oz.Handle(1 << 28, **flags)
    want = y0.copy()
    getattr(h, "scsrmv" if single else "csrmv")(m, n, nnz, one(1.25), val, colind, rowptr, x, one(-0.5), want)
    say(f"csr many slices {prec} {m}x{n} {flags} bad={bad}")
    for _ in range(2):
        y = dev(y0)
        getattr(H, prec + "csrmv")(m, n, nnz, 1.25, dev(val), dev(colind), dev(rowptr), dev(x), -0.5, y)
        got = host(y)
        assert (H.nSplitA, H.nSplitB) == (h.nSplitA, h.nSplitB)
        assert np.array_equal(np.isfinite(got), np.isfinite(want))
        ok = np.isfinite(want)
        assert bits_equal(got[ok], want[ok]), first_diff(got[ok], want[ok])
