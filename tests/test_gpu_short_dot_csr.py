"""The one-workgroup DOT (n <= 8192) and the row-block kernels of the sparse split and product at the
edges of their sizes, bitwise against the oracle: vectors around each kernel instance's length and the
hand-over to the general path, slice counts and flags, rows that end a block, blocks whose nonzeros
exceed the stage, empty rows, and more matrix slices than the narrow stage holds."""
import numpy as np
import pytest

from gpu_util import bits_equal, dev, first_diff, host, say, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    torch_cuda()
    import ozblas_amd
    return ozblas_amd


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 256, 1023, 1024, 1025, 4095, 4096, 4097, 8191, 8192, 8193])
@pytest.mark.parametrize("flags", [dict(sumMode=1), dict(sumMode=0), dict(sumMode=1, reproMode=0),
                                   dict(sumMode=1, nSplitMax=3, reproMode=1), dict(sumMode=0, nSplitMax=1)],
                         ids=lambda f: ",".join(f"{k}={v}" for k, v in f.items()))
def test_short_dot_bitwise(oz, oracle, n, flags):
    H = oz.Handle(1 << 28, **flags)
    say(f"short dot n={n} {flags}")
    for phi in (0.5, 2.0, 12.0):  # phi = 12: more than 8 slices, the general path
        x, y = oracle.init_mat(n, 1, n, phi, 2, 41), oracle.init_mat(n, 1, n, 0.5, 2, 42)
        h = oracle.Handle(1 << 30, **flags)
        want = h.dot(n, x, y)
        dx, dy = dev(x), dev(y)
        for _ in range(2):  # the second call meets the scratch the first one left
            assert np.float64(H.ddot(n, dx, dy)).view(np.uint64) == np.float64(want).view(np.uint64), phi
            assert (H.nSplitA, H.nSplitB) == (h.nSplitA, h.nSplitB)
        assert np.float64(H.ddot(n, dx, dx)).view(np.uint64) == \
            np.float64(oracle.Handle(1 << 30, **flags).dot(n, x, x)).view(np.uint64)
    z = np.zeros(n)
    assert H.ddot(n, dev(z), dev(z)) == oracle.Handle(1 << 30, **flags).dot(n, z, z)
    z[n - 1] = np.inf
    assert np.isnan(H.ddot(n, dev(z), dev(z))) == np.isnan(oracle.Handle(1 << 30, **flags).dot(n, z, z))


@pytest.mark.parametrize("n", [700, 5000])
def test_short_sdot_bitwise(oz, oracle, n):
    x, y = oracle.s_init_mat(n, 1, n, 1.0, 2, 43), oracle.s_init_mat(n, 1, n, 1.0, 2, 44)
    for mode in (0, 1):
        want = np.float32(oracle.Handle(1 << 30, sumMode=mode).sdot(n, x, y))
        say(f"short sdot n={n} sumMode={mode}")
        got = np.float32(oz.Handle(1 << 28, sumMode=mode).sdot(n, dev(x), dev(y)))
        assert got.view(np.uint32) == want.view(np.uint32)


def _rows(lengths, seed, phi, oracle):
    n = len(lengths)
    rng = np.random.RandomState(seed)
    rowptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    nnz = int(rowptr[-1])
    colind = rng.randint(0, n, nnz).astype(np.int32)
    return n, nnz, rowptr, colind, oracle.init_mat(max(nnz, 1), 1, max(nnz, 1), phi, 2, seed)[:nnz]


CASES = {
    "one_row": [5],
    "block": [7] * 256,
    "block_plus_one": [7] * 257,
    "stage_full": [8] * 256 + [3] * 40,         # 2048 nonzeros in the first block
    "stage_over": [9] * 256 + [2] * 300,        # the first block passes through the stage in parts
    "empty_rows": [0, 3] * 300,
    "all_empty": [0] * 300,
    "long_row": [2] * 100 + [3000] + [1] * 500,
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("sumMode,phi", [(1, 0.5), (0, 1.0), (1, 6.0)])
@pytest.mark.parametrize("presplit", [False, True])
def test_csr_row_blocks_bitwise(oz, oracle, name, sumMode, phi, presplit):
    n, nnz, rowptr, colind, val = _rows(CASES[name], 51, phi, oracle)
    if nnz == 0 and presplit:
        pytest.skip("nothing to split")
    x = oracle.init_mat(n, 1, n, phi, 2, 52)
    y0 = oracle.init_mat(n, 1, n, 1.0, 2, 53)
    h = oracle.Handle(1 << 30, sumMode=sumMode)
    want = y0.copy()
    say(f"csr blocks {name} sumMode={sumMode} phi={phi} presplit={presplit}")
    H = oz.Handle(1 << 28, sumMode=sumMode)
    dval, dcol, drow, dx, dy = dev(val if nnz else np.zeros(1)), dev(colind if nnz else np.zeros(1, np.int32)), \
        dev(rowptr), dev(x), dev(y0)
    if presplit:
        hA = h.csrmv_splitA(n, n, nnz, val, rowptr)
        A = H.dcsrmv_splitA(n, n, nnz, dval, drow)
        assert (H.nSplitA_, H.splitShift) == (h.nSplitA_, h.splitShift)
    else:
        A, hA = dval, val
    h.csrmv(n, n, nnz, 1.25, hA, colind, rowptr, x, -0.5, want)
    H.dcsrmv(n, n, nnz, 1.25, A, dcol, drow, dx, -0.5, dy)
    got = host(dy)
    assert bits_equal(got, want), first_diff(got, want)
