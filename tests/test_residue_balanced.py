"""CPU check of the residue writers' arithmetic (res_group, res_member_byte / res_member_float of
ozblas_amd/csrc/oz_residue.hpp), restated in IEEE binary64 / binary32 with the library's own constants,
against exact integers: the group representative nearest zero, and each member's balanced residue from
one binary32 fused multiply-add, at the values next to the rounding boundaries for every modulus."""
import random
from fractions import Fraction as Fr

import numpy as np
import pytest

from test_residue_model import MAXMOD, rc  # noqa: F401  (the library's constants, a fixture)

MAGIC = 12582912


def fma64(a, b, c):
    return float(Fr(float(a)) * Fr(float(b)) + Fr(float(c)))


def group(sf, P, inv, pw2):
    q = np.rint(np.float64(sf) * inv)
    r0 = fma64(-q, P, sf)
    assert int(r0) == int(sf) - int(q) * int(P) and abs(r0) <= P / 2 + 2
    x = np.float64(r0) * np.float64(pw2)
    assert abs(x) < 2.0 ** 53 and int(x) == int(r0) * int(pw2)
    q = np.rint(x * inv)
    return int(fma64(-q, P, x))


def member(rx, p, invpf):
    assert abs(rx) <= 1 << 23 and int(np.float32(rx)) == rx
    v = Fr(rx) * Fr(float(invpf)) + MAGIC      # one rounding, to integers: [2^23, 2^24)
    assert (1 << 23) <= v < (1 << 24)
    q = round(v) - MAGIC                        # Python rounds halves to even, as binary32 does
    bits = (0x4B400000 + q) & 0xFFFFFFFF
    s24 = ((bits & 0xFFFFFF) ^ 0x800000) - 0x800000  # the 24-bit operand, sign-extended
    byte = (rx - s24 * p) & 0xFF
    flt = float(np.float32(fma64(-q, p, rx)))
    return byte, flt


def test_group_and_member_residues(rc):  # noqa: F811
    c, _ = rc[MAXMOD]
    rng = random.Random(3)
    for t in range(MAXMOD):
        p, g = int(c["p"][t]), t // 3
        P, inv, invpf = int(c["Pg"][g]), c["invPg"][g], c["invpf"][t]
        assert P < 1 << 24
        # representatives around every boundary: k p + (p +- 1) / 2 next to the ends and in between
        edge = P // 2
        reps = {0, 1, -1, edge, -edge, edge - 1, 1 - edge}
        for k in [0, 1, edge // p - 1, edge // p - 2] + [rng.randrange(0, max(1, edge // p)) for _ in range(40)]:
            for d in (p // 2 - 1, p // 2, p // 2 + 1, p // 2 + 2):
                reps |= {k * p + d, -(k * p + d)}
        for rx in reps:
            if abs(rx) > edge:
                continue
            byte, flt = member(rx, p, invpf)
            r = ((byte ^ 0x80) - 0x80)
            assert (r - rx) % p == 0 and -128 <= r <= 127 and (p == 256 or abs(r) <= (p - 1) // 2), (p, rx)
            assert (int(flt) - rx) % p == 0 and abs(flt) <= p / 2, (p, rx)
        # group representatives at the edges of the significand and of the shift table
        for sh in (0, 1, 29, 511):
            for f in [1, 3, (1 << 53) - 1, (1 << 52) + 1, P, P // 2, P // 2 + 1] + \
                    [rng.getrandbits(53) for _ in range(6)]:
                for sf in (f, -f):
                    rx = group(sf, float(P), inv, int(c["pow2g"][g][sh]))
                    assert abs(rx) <= (P + 1) // 2 <= 1 << 23 and (rx - sf * pow(2, sh, P)) % P == 0


@pytest.mark.parametrize("lowest", [255, 253])
def test_binary32_reciprocal_margin(rc, lowest):  # noqa: F811
    """The margin the quotient relies on: the relative error of RN(1/p) is below 2^-24 for every odd p."""
    c, _ = rc[MAXMOD]
    for t in range(MAXMOD):
        p = int(c["p"][t])
        if p % 2 and p <= lowest:
            assert abs(Fr(float(c["invpf"][t])) * p - 1) < Fr(1, 1 << 24)
