"""CPU check of the clear-cut case of NearSum (SumCert of ozblas_amd/csrc/oz_nearsum.hpp, host build):
whenever it settles a sum, the value is the exact sum rounded to nearest even (exact rationals) -- for
random values, cancellation, near ties, powers of two, and values outside its range, which it must
leave to the full algorithm."""
import ctypes
import os
import random
from fractions import Fraction as Fr

import numpy as np

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ozblas_amd", "libozblas_mi355x.so")


def cert(v):
    f = ctypes.CDLL(LIB).ozblas_internal_sum_cert
    f.restype = ctypes.c_int32
    a = np.array(v, dtype=np.float64)
    t = ctypes.c_double()
    return t.value if f(len(v), a.ctypes.data_as(ctypes.c_void_p), ctypes.byref(t)) else None


def test_certified_sums_are_correctly_rounded():
    rng = random.Random(8)
    settled = 0
    for trial in range(6000):
        n = rng.randint(1, 32)
        spread = rng.choice([1, 8, 40, 90])
        v = [rng.uniform(-1, 1) * 2.0 ** rng.randint(-spread, spread) for _ in range(n)]
        kind = trial % 6
        if kind == 1:  # cancellation
            v += [-x for x in v[: n // 2]]
        elif kind == 2:  # a tie or next to one
            x = float(rng.getrandbits(52) | (1 << 52))
            v = [x, 0.5, rng.choice([0.0, 2.0 ** -60, -(2.0 ** -60), 2.0 ** -110])]
        elif kind == 3:  # at a power of two
            v = [2.0 ** rng.randint(-5, 5), rng.choice([-1, 1]) * 2.0 ** -rng.randint(50, 60)]
        want = float(sum(Fr(x) for x in v))
        got = cert(v)
        if got is not None:
            settled += 1
            assert got == want, (v, got, want)
    assert settled > 3000


def test_left_to_the_full_algorithm():
    inf, nan = float("inf"), float("nan")
    for v in ([0.0], [1.0, -1.0], [inf], [nan, 1.0], [inf, -inf], [2.0 ** 900], [2.0 ** 900, 1.0, -2.0 ** 900],
              [2.0 ** -910 * 1.5], [4.0], [float((1 << 52) + 1), 0.5]):
        assert cert(v) is None, v
