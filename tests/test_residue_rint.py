"""The prep kernel's residue quotient, q = rint(u / p) from one float32 fma with 1.5 2^23, checked on
the CPU over every u the byte dot products can produce and every modulus: the low byte of
u - (2^22 + q) p is that of sym(u mod p)."""
import numpy as np
import pytest

from test_residue_arith import MODULI, _quotient


@pytest.mark.parametrize("p", MODULI)
def test_rint_quotient_exhaustive(p):
    u = np.arange(-(1 << 16), (1 << 19) + (1 << 16), dtype=np.int64)
    ipf = np.float64(np.float32(1.0 / p))
    if p % 2:
        assert np.abs(np.abs(u * ipf - np.floor(u * ipf)) - 0.5).min() > 2.0 ** -10
    low = _quotient(u, p)
    r = u - low * p
    s = u % p
    s = np.where(s > p - 1 - p // 2, s - p, s)
    assert np.array_equal(r & 0xFF, s & 0xFF)
    assert (low < 1 << 23).all()                              # positive as a signed 24-bit number
