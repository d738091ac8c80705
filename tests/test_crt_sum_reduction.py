"""The residue products' reduction of an int32 sum mod an odd modulus, restated in IEEE float32:
f - m rint(f fl(1/m)) with f = h (2^19 mod m) + l of v = h 2^19 + l. It is the symmetric residue
for every modulus of the scheme, at the sums nearest to a half-integer quotient over the whole
range, at the range's ends and in between."""
import numpy as np
import pytest

MODULI = [255, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197, 193, 191, 181, 179, 173]


@pytest.mark.parametrize("m", MODULI)
def test_symmetric_residue(m):
    c = (1 << 19) % m
    c = c - m if 2 * c > m else c
    rng = np.random.default_rng(m)
    top = 2 ** 31 - 128
    q = rng.integers(-(top // m), top // m, 200000)
    v = np.concatenate([q * m + (m - 1) // 2, q * m - (m - 1) // 2, rng.integers(-top, top, 200000),
                        np.arange(-70000, 70000), np.arange(top - 1000, top), np.arange(-top, -top + 1000)])
    v = v[np.abs(v) <= top]
    f = ((v >> 19) * c + (v & 0x7FFFF))
    assert np.abs(f).max() < 2 ** 20
    f32 = f.astype(np.float32)
    quot = np.rint(f32 * np.float32(1.0 / m)).astype(np.int64)  # one rounding of 1 / m, one of the product
    r = f - quot * m
    want = (v + (m - 1) // 2) % m - (m - 1) // 2
    assert np.array_equal(r, want)
