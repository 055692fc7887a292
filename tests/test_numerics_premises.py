"""Numerical premises of the device arithmetic, checked on the CPU in numpy.

The kernels rely on two facts about IEEE rounding that no GPU test could
isolate: (1) for a power-of-two scale, the low FP16 part of a split formed by
one rounding of the exact a * scale - hi (an FMA) equals the two-step form
fp16(fp32(a * scale) - hi); (2) a BF16 value widened to FP16 is exact from
2^-14 (FP16's smallest normal number) up, and within 2^-25 below.
"""
import subprocess

import numpy as np
import pytest


def _split_two_step(a, scale):
    v = (a * scale).astype(np.float32)
    hi = v.astype(np.float16)
    lo = (v - hi.astype(np.float32)).astype(np.float16)
    return hi, lo


def _split_fma(a, scale):
    v = (a * scale).astype(np.float32)
    hi = v.astype(np.float16)
    exact = a.astype(np.float64) * float(scale) - hi.astype(np.float64)  # exact in FP64
    return hi, exact.astype(np.float16)  # one rounding, as the FMA's


def test_fma_low_part_equals_the_two_step_split():
    rng = np.random.default_rng(0)
    # accumulators of taps scaled into [2^14, 2^15): sums up to a few times 2^15
    a = np.concatenate([rng.uniform(0, 2 ** 16, 200000), rng.uniform(0, 1e-3, 50000),
                        np.float32([0.0, 1.0, 2 ** 15, 65535.0])]).astype(np.float32)
    for s in (14, 15, 16, 20):
        scale = np.float32(2.0 ** -s)
        h1, l1 = _split_two_step(a, scale)
        h2, l2 = _split_fma(a, scale)
        assert np.array_equal(h1.view(np.uint16), h2.view(np.uint16))
        assert np.array_equal(l1.view(np.uint16), l2.view(np.uint16))


def test_the_fma_check_sees_a_double_rounding():
    """The same comparison with a scale that is not a power of two (the
    product then rounds before the subtraction) finds differences."""
    rng = np.random.default_rng(1)
    a = rng.uniform(0, 2 ** 16, 200000).astype(np.float32)
    scale = np.float32(1.0 / 3.0)
    _, l1 = _split_two_step(a, scale)
    _, l2 = _split_fma(a, scale)
    assert not np.array_equal(l1.view(np.uint16), l2.view(np.uint16))


def test_bf16_widens_to_fp16():
    # every BF16 bit pattern of a finite value in [0, 65504]
    bits = np.arange(0, 0x7F80, dtype=np.uint32)
    v = (bits << 16).view(np.float32)
    v = v[v <= 65504.0]
    h = v.astype(np.float16).astype(np.float32)
    normal = v >= 2.0 ** -14
    assert np.array_equal(h[normal], v[normal])
    assert np.abs(h[~normal] - v[~normal]).max() <= 2.0 ** -25


def test_reciprocal_and_residual_divide_like_float64():
    """The histogram bins divide with q0 = x r, q = q0 + (x - q0 d) r for the
    correctly rounded r = 1/d (two FMAs): the correctly rounded quotient x / d
    for every d whose significand is not all ones."""
    from fractions import Fraction

    def fma(a, b, c):
        return float(Fraction(a) * Fraction(b) + Fraction(c))  # one rounding

    rng = np.random.default_rng(9)
    pairs = [(0.1, 60000.7), (1.0, 40000.0), (1.0, 65535.0), (13333.0, 26666.0), (0.0, 65535.0)]
    pairs += [tuple(sorted(rng.uniform(0, 65535, 2))) for _ in range(10)]
    for lo, hi in pairs:
        d = hi - lo
        r = 1.0 / d
        for v in rng.integers(1, 65536, 300).astype(float):
            x = v - lo
            q0 = x * r
            assert fma(fma(-q0, d, x), r, q0) == x / d


def test_rings_hold_at_most_seven_pixels_per_radius():
    """A ring floor(sqrt(dx^2 + dy^2)) = r holds at most 7 (r + 1) lattice
    points: the bound that keeps the 16-bit radius counters from overflowing."""
    R = 3000
    x = np.arange(-R, R + 1, dtype=np.int64)
    count = np.zeros(R + 1, np.int64)
    for y in range(R + 1):
        r = np.floor(np.sqrt((x * x + y * y).astype(np.float64))).astype(np.int64)
        count += np.bincount(r[r <= R], minlength=R + 1) * (1 if y == 0 else 2)
    assert (count <= 7 * (np.arange(R + 1) + 1)).all()


def _quick_quotient(x, d):
    """x / d as the kernels divide by a shared divisor: the rounded reciprocal,
    a product and one residual, each rounded to float32 (the fused products
    formed in 64-bit significands)."""
    r = np.float32(1.0) / d
    q = x * r
    e = (x.astype(np.float64) - q.astype(np.float64) * np.float64(d)).astype(np.float32)  # exact in FP64
    return (e.astype(np.longdouble) * np.longdouble(r) + q.astype(np.longdouble)).astype(np.float32)


def test_float32_division_by_a_shared_divisor():
    """Every dividend significand against divisors about the ends of their
    binade, fractions and maxima of fields; and whole numbers below 2^16 against
    whole ones, as the field combination divides."""
    x = np.arange(1 << 23, 1 << 24, dtype=np.uint32).astype(np.float32)
    for d in (1.0, 3.0, 0.7, 65535.0, np.float32(2.0) - np.float32(2.0 ** -22), np.float32(1.0) + np.float32(2.0 ** -23)):
        d = np.float32(d)
        assert np.array_equal(_quick_quotient(x, d), x / d), d
    whole = np.arange(0, 65536, dtype=np.float32)
    rng = np.random.default_rng(5)
    for d in np.concatenate([[1, 2, 3, 32767, 32768, 65534, 65535], rng.integers(4, 65534, 100)]):
        assert np.array_equal(_quick_quotient(whole, np.float32(d)), whole / np.float32(d)), d


def test_square_root_from_the_reciprocal_root():
    """The distance transform's square root of a whole number (one residual on
    x times the reciprocal square root) is the rounded one for reciprocal roots
    one unit in the last place to either side, the instruction's bound: all
    numbers up to 2^20, and samples up to the largest squared distance."""
    rng = np.random.default_rng(6)
    top = 3 * 4095 ** 2
    n = np.concatenate([np.arange(1, 1 << 20), rng.integers(1 << 20, top, 1_500_000), np.arange(top - 1000, top + 1),
                        np.arange(1, 4096) ** 2, np.arange(2, 4096) ** 2 - 1, np.arange(1, 4096) ** 2 + 1])
    x = n.astype(np.float32)  # the kernel's conversion rounds above 2^24
    want = np.sqrt(x)
    mid = (1.0 / np.sqrt(x.astype(np.float64))).astype(np.float32)
    for y in (mid, np.nextafter(mid, np.float32(0)), np.nextafter(mid, np.float32(2))):
        g = x * y
        r = (x.astype(np.float64) - g.astype(np.float64) ** 2).astype(np.float32)  # exact in FP64
        got = (r.astype(np.longdouble) * (np.float32(0.5) * y).astype(np.longdouble) + g.astype(np.longdouble))
        assert np.array_equal(got.astype(np.float32), want)


EVERY_VALUE = r"""
#include <cmath>
#include <cstdio>
int main() {
    static float top[65536];
    for (int i = 0; i < 65536; ++i) top[i] = (float)i;
    long long bad = 0;
    for (int i = 1; i < 65536; ++i) {  // combine: x / d of 16-bit whole numbers
        const float d = (float)i, r = 1.0f / d;
        int wrong = 0;
        for (int j = 0; j < 65536; ++j) {
            const float x = top[j], q = x * r;
            wrong += __builtin_fmaf(__builtin_fmaf(-q, d, x), r, q) != x / d;
        }
        bad += wrong;
    }
    std::printf("%lld\n", bad);
    for (int n = 1; n <= 3 * 4095 * 4095; ++n) {  // the distance transform's root
        const float x = (float)n, mid = (float)(1.0 / std::sqrt((double)x)), want = std::sqrt(x);
        for (int ulp = -1; ulp <= 1; ++ulp) {
            const float y = ulp == 0 ? mid : std::nextafter(mid, ulp < 0 ? 0.0f : 2.0f), g = x * y;
            if (__builtin_fmaf(__builtin_fmaf(-g, g, x), 0.5f * y, g) != want) std::printf("%d:%d\n", n, ulp);
        }
    }
}
"""


DECIDED_BY_SEED = {8259749: [1], 13440042: [-1], 14344251: [-1], 15635314: [-1, 1], 33038995: [1], 33038996: [1],
                   33038997: [1]}


def test_every_whole_quotient_and_root(tmp_path):
    """All quotients of 16-bit whole numbers, and all roots up to the largest
    squared distance.  With the rounded reciprocal root every root is the rounded
    one; with a neighbour of it, as the instruction may return, all but those of
    DECIDED_BY_SEED, which the GPU tests compare (the last three are 4 times the
    first and its neighbours that round to the same float32)."""
    with open("/proc/cpuinfo") as f:
        if " fma " not in f.read():
            pytest.skip("no fused multiply-add on this CPU: too slow in software")
    src, exe = tmp_path / "every.cpp", tmp_path / "every"
    src.write_text(EVERY_VALUE)
    subprocess.run(["g++", "-std=c++17", "-O3", "-mavx2", "-mfma", "-ffp-contract=off", "-fno-math-errno", str(src),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, check=True).stdout.split()
    assert out == ["0"] + [f"{n}:{ulp}" for n, ulps in DECIDED_BY_SEED.items() for ulp in ulps]
