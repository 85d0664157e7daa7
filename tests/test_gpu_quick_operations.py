"""The bit-exact build's quick reciprocal, quotient and square root round as the
IEEE operations: every binary32 significand (and exponent parity, of a root),
every pair of significands whose quotient lies close enough to a rounding
midpoint to be in doubt, operands over the whole range the callers accept, and
binary64 reciprocals of random significands and of those from all ones down."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ONE = np.uint32(0x3f800000)


def same(got, ref, *operands):
    bad = np.flatnonzero(got.view(f"u{got.itemsize}") != ref.view(f"u{ref.itemsize}"))
    assert bad.size == 0, (bad.size, [tuple(float(o[i]).hex() for o in operands) for i in bad[:4]])


def random32(rng, n, lo, hi):
    """significands at random, exponents lo .. hi - 1"""
    e = rng.integers(lo + 127, hi + 127, n).astype(np.uint32)
    return ((e << np.uint32(23)) | rng.integers(0, 1 << 23, n).astype(np.uint32)).view(np.float32)


def test_reciprocals(mpcf):
    print("[quick] reciprocals", flush=True)
    b = (ONE + np.arange(1 << 23, dtype=np.uint32)).view(np.float32)
    same(mpcf.test_quotient("rcp", b=b), np.float32(1) / b, b)
    # densities, G and wave speeds from 2^-40, sums of weights up to 2^43
    b = random32(np.random.default_rng(1), 1 << 21, -90, 80)
    same(mpcf.test_quotient("rcp", b=b), np.float32(1) / b, b)


def test_roots(mpcf):
    print("[quick] roots", flush=True)
    a = (ONE + np.arange(1 << 24, dtype=np.uint32)).view(np.float32)     # 1 <= a < 4
    same(mpcf.test_quotient("sqrt", a=a), np.sqrt(a), a)
    a = random32(np.random.default_rng(2), 1 << 21, -80, 81)
    same(mpcf.test_quotient("sqrt", a=a), np.sqrt(a), a)


def close_pairs(scale, reach):
    """all 24-bit significands a, b for which 2^scale a - m b = r, m odd, |r| <= reach:
    the quotient is r / (2^scale b) off a midpoint m / 2^scale.  An odd b needs an
    odd r; of b = 2^k b', r = 2^k r' with r' odd, and the equation divided by 2^k"""
    for k in range(int(reach).bit_length()):
        b = (np.arange(max(1, 1 << (22 - k)), dtype=np.int64) * 2 + 1) + (1 << (23 - k))   # odd, k bits shorter
        x = np.ones_like(b)                                    # 2^-(scale - k) modulo b
        for _ in range(scale - k):
            x = np.where(x & 1, x + b, x) >> 1
        for r in range(1, (reach >> k) + 1, 2):
            for sign in (1, -1):
                a = (sign * r * x) % b
                for shift in range(1 << (k + 1)):              # a in [2^23, 2^24) of that residue
                    aa = a + shift * b
                    ok = (aa >= 1 << 23) & (aa < 1 << 24)
                    # scale 24: quotients in [1, 2); 25: in [1/2, 1)
                    ok &= (aa >= b << k) if scale == 24 else (aa < b << k)
                    if ok.any():
                        yield aa[ok], (b << k)[ok], sign * (r << k)


def test_quotients_next_to_midpoints(mpcf):
    """before its last rounding the quick quotient is within 2.25 2^-24 units in
    the last place of the exact one: 4.5 of the residues r above"""
    pairs = 0
    for scale in (24, 25):
        print("[quick] quotients", scale, flush=True)
        for a, b, r in close_pairs(scale, 5):
            if pairs == 0:                                     # the construction itself, exactly
                m = ((1 << scale) * a - r) // b
                assert np.array_equal(m * b + r, (1 << scale) * a) and (m & 1).all()
            a, b = (x.astype(np.float32) for x in (a, b))
            same(mpcf.test_quotient("div", a=a, b=b), a / b, a, b)
            pairs += a.size
    assert pairs > 1 << 24, pairs


def test_quotients_of_every_magnitude(mpcf):
    print("[quick] magnitudes", flush=True)
    rng = np.random.default_rng(3)
    a, b = random32(rng, 1 << 22, -80, 81), random32(rng, 1 << 22, -40, 41)
    a = a * rng.choice(np.float32([1, -1]), a.size)
    keep = np.abs(np.log2(np.abs(a, dtype=np.float64)) - np.log2(b, dtype=np.float64)) < 81
    a, b = a[keep], b[keep]
    same(mpcf.test_quotient("div", a=a, b=b), a / b, a, b)


def test_binary64_reciprocals(mpcf):
    print("[quick] binary64", flush=True)
    rng = np.random.default_rng(4)
    one = np.uint64(0x3ff << 52)
    b = (one + rng.integers(0, 1 << 52, 1 << 23).astype(np.uint64)).view(np.float64)
    same(mpcf.test_quotient("rcp64", b=b), 1 / b, b)
    # just below two, from the significand of all ones down
    b = (one + (np.uint64(1) << np.uint64(52)) - np.uint64(1) - np.arange(1 << 16, dtype=np.uint64)).view(np.float64)
    same(mpcf.test_quotient("rcp64", b=b), 1 / b, b)
    # ten squared indicators, as the weights take them
    i = np.float64(random32(rng, 1 << 23, -20, 60))
    b = 10.0 * i * i
    same(mpcf.test_quotient("rcp64", b=b), 1 / b, b)
