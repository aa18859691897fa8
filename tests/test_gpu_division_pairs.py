"""The shortened division (div_inrange) against '/' on the operands where a
slightly less exact reciprocal would show: divisors 2 - j*2^-52 with j < 2^33,
whose reciprocals lie next to the midpoint of two doubles, and numerators that
put the quotient next to one.  Random mantissas do not meet them."""
import numpy as np
import pytest

from test_gpu_division import doubles, run, same_bits

pytestmark = pytest.mark.gpu

# (mantissa of a, j), from an enumeration of every odd j below 2^36: quotients
# that come out as the neighbouring double when the reciprocal is refined to
# 2^-73 by one step instead of by two Newton steps
PAIRS = np.array([
    (0x865586dd92f9, 0x2bd15b85), (0x146d298b11a31, 0x31f5c159), (0x19d79af0e5a51, 0x5adcce7d),
    (0x1e4bbcc977aba, 0xffffff3), (0x276276276275b, 0xd), (0x2904c524b73a3, 0x73ee561b),
    (0x2c3f3522c3f3b, 0xffffff7), (0x386b203def3d2, 0x24a91d59), (0x3f96f06ad9e15, 0x9497e809),
    (0x4053b8c4f89d1, 0x39b05653), (0x4ebe258bfec55, 0x1cd82b31), (0x535056d46796c, 0xb504f2d),
    (0x59488c3e9b089, 0x6e45ba9b), (0x5feef7135daed, 0xbffffdbf), (0x620ce4e284f57, 0x2991b83f),
    (0x67d71f530317e, 0x5faa840b), (0x71c71c0e38e3b, 0x7fffffd), (0x786f9256caa46, 0x38918bcb),
    (0x86acfb91b48a0, 0x1fffffeb), (0x896b1c48f1c8a, 0x6712a1b3), (0x8e12a4f8b96f1, 0x59ccbdb5),
    (0x9419623f7898e, 0x17fffff5), (0xa40d8617e9116, 0xddb3d67), (0xad0a1a7dd2180, 0x478dde1d),
    (0xaecde01f1dde6, 0x3c660f5d), (0xb450531fca1c9, 0x7d38444b), (0xb5cc4b3fb7470, 0x16a09e5d),
    (0xbb457c92798a9, 0x24a91d5b), (0xc5f34b1456972, 0x152a7fa1), (0xccd44e8d5c0cb, 0x265ddcd1),
    (0xd0d7516cd5a84, 0x4eca7593), (0xd4a7fbaf0df22, 0x7aa33ded),
], dtype=np.uint64)


def test_hard_pairs(hipdev):
    """Every pair, both signs, with exponents over div_inrange's range."""
    rng = np.random.default_rng(21)
    reps = 512
    ma = np.tile(PAIRS[:, 0], reps)
    mb = np.uint64(1 << 52) - np.tile(PAIRS[:, 1], reps)
    eb = rng.integers(-1000, 999, size=mb.size)
    ea = np.clip(eb + rng.integers(-760, 761, size=mb.size), -960, 999)
    eb[: len(PAIRS)] = ea[: len(PAIRS)] = 0
    a = doubles(rng, ea, ma) * np.where(rng.random(ma.size) < 0.5, -1.0, 1.0)
    b = doubles(rng, eb, mb)
    qf, qi = run(hipdev, 0, a, b)
    bad = ~same_bits(qf, qi)
    assert not bad.any(), (bad.sum(), a[bad][:4], b[bad][:4], qf[bad][:4], qi[bad][:4])


@pytest.mark.parametrize("p", [1, 2])
def test_weights_of_scaled_indicators(hipdev, p):
    """The indicators are held times 4, so a weight's operands reach 2^169."""
    rng = np.random.default_rng(22 + p)
    n = 1 << 20
    b = doubles(rng, rng.integers(-148, 169, size=n))
    t = doubles(rng, rng.integers(-380, 169, size=n))
    mb = np.uint64(1 << 52) - rng.choice(PAIRS[:, 1], size=n // 4)
    b[: n // 4] = doubles(rng, rng.integers(-148, 169, size=n // 4), mb)
    t[: n // 4] = doubles(rng, rng.integers(-148, 169, size=n // 4), rng.choice(PAIRS[:, 0], size=n // 4))
    qf, qi = run(hipdev, p, t, b)
    assert same_bits(qf, qi).all()
