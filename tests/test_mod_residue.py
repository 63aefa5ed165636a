"""CPU check of the product kernels' reduction modulo p (mod_residue of ozblas_amd/csrc/oz_digits.hpp, host
build): the canonical residue for every modulus of the list, at multiples of p and their neighbours, at the largest
sums that 65536 products of balanced residues give, and at random."""
import ctypes
import os

import numpy as np

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ozblas_amd", "libozblas_mi355x.so")


def moduli():
    out = [256]
    for p in range(255, 2, -1):
        if all(np.gcd(p, q) == 1 for q in out):
            out.append(p)
    return out


def test_canonical_residue_of_every_modulus():
    f = ctypes.CDLL(LIB).ozblas_internal_mod_residue
    rng = np.random.default_rng(3)
    for p in moduli() + [3, 5, 7]:
        half = p // 2
        top = half * half * 65536
        mult = np.unique(np.concatenate([rng.integers(-(top // p), top // p + 1, 20000),
                                         np.arange(-300, 301), top // p - np.arange(300), np.arange(300) - top // p]))
        v = np.concatenate([p * mult + d for d in (-2, -1, 0, 1, 2)] + [rng.integers(-top, top + 1, 20000),
                                                                        np.array([top, -top, 0])])
        v = v[np.abs(v) <= top].astype(np.int32)
        out = np.empty(len(v), dtype=np.uint8)
        f(ctypes.c_int32(len(v)), v.ctypes.data_as(ctypes.c_void_p), ctypes.c_int32(p),
          out.ctypes.data_as(ctypes.c_void_p))
        assert np.array_equal(out, (v.astype(np.int64) % p).astype(np.uint8)), p
