"""The drift kernels' short forms of exact operations on the device, bit for bit
against the IEEE operation or the oracle over the ranges they are used in:
every float for the square root and the rounding of a draw; random operands,
the edges of the range and quotients next to a rounding midpoint for the
quotient; and the whole clamped draw."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CHUNK = 1 << 24


def every_float(lo_bits, hi_bits):
    for b in range(lo_bits, hi_bits, CHUNK):
        yield np.arange(b, min(b + CHUNK, hi_bits), dtype=np.uint32).view(np.float32)


def bits_of(x):
    return int(np.float32(x).view(np.uint32))


# four parts of 2^-96 .. the largest float
@pytest.mark.parametrize("part", range(4))
def test_sqrt_pos_every_float(gpu, part):
    lo, hi = bits_of(2.0 ** -96), 0x7f800000
    step = (hi - lo + 3) // 4
    for x in every_float(lo + part * step, min(lo + (part + 1) * step, hi)):
        assert np.array_equal(gpu.device_math("sqrt_pos", x).view(np.uint32), np.sqrt(x).view(np.uint32)), x[0]


def counts(oracle, v, top):
    """round half away from zero of v clamped to [0, top], NaN to 0"""
    return oracle.f2i(oracle.round_away(np.where(np.isnan(v), np.float32(0), np.clip(v, np.float32(0), np.float32(top)))))


# four parts of 0 .. infinity, and the first NaN
@pytest.mark.parametrize("part", range(4))
def test_round_count_every_float(gpu, oracle, part):
    top = np.float32(2147483520)
    step = 0x7f800002 // 4 + 1
    for v in every_float(part * step, min((part + 1) * step, 0x7f800002)):
        assert np.array_equal(gpu.device_math("round_count", v, top), counts(oracle, v, top)), v[0]


def test_round_count_clamps(gpu, oracle):
    rng = np.random.default_rng(21)
    n = 1 << 20
    top = rng.integers(1, 1 << 22, n).astype(np.float32)
    v = (top * rng.uniform(-0.2, 1.2, n)).astype(np.float32)
    v[::7] = np.rint(v[::7] * 2) / 2
    v[:12] = [np.nan, -np.nan, np.inf, -np.inf, -0.0, -0.25, -0.5, -0.75, -3e9, 3e9, 1e38, -1e38]
    v[12:24], v[24:36] = top[12:24] + np.float32(0.5), top[24:36] - np.float32(0.5)
    assert np.array_equal(gpu.device_math("round_count", v, top), counts(oracle, v, top))


@pytest.mark.parametrize("kind", ["random", "edges", "midpoints"])
def test_div_mid(gpu, kind):
    rng = np.random.default_rng(22)
    for _ in range(8):
        n = 1 << 21
        den = np.exp2(rng.uniform(-20, 20, n)).astype(np.float32)
        num = np.exp2(rng.uniform(-80, 20, n)).astype(np.float32)
        if kind == "random":   # the kernels' own: den in [1/2, 3/2], num below 3/2
            den[::2] = rng.uniform(0.5, 1.5, n // 2)
            num[::4] = rng.uniform(0.0, 1.5, n // 4)
            num[1::4] = den[1::4] * np.float32(1) + rng.uniform(-1e-6, 1e-6, n // 4).astype(np.float32)
        elif kind == "edges":
            ends = np.array([2.0 ** -80, 2.0 ** -79, 2.0 ** -20, 0.5, 1.0, 1.5, 2.0 ** 20, 0.0], np.float32)
            num[::2] = rng.choice(ends, n // 2)
            den[1::3] = rng.choice(ends[2:7], len(den[1::3]))
            near = np.array([-2, -1, 0, 1, 2])
            ok = num > 0
            num[ok] = (num.view(np.int32)[ok] + rng.choice(near, ok.sum()).astype(np.int32)).view(np.float32)
        else:                  # num = RN(den m), m half way between two floats
            m = 1.0 + rng.integers(0, 1 << 23, n) * 2.0 ** -23 + 2.0 ** -24
            m *= np.exp2(rng.integers(-60, 1, n))
            num = (den.astype(np.float64) * m).astype(np.float32)
        num = np.clip(num, 0, np.float32(2.0 ** 20))
        num[(num > 0) & (num < np.float32(2.0 ** -80))] = np.float32(2.0 ** -80)
        num[::5] = -num[::5]
        den[::3] = -den[::3]
        got, want = gpu.device_math("div_mid", num, den), num / den
        nonzero = num != 0     # the sign of a zero is no one's concern: it becomes a mean of 0
        assert np.array_equal(got[nonzero].view(np.uint32), want[nonzero].view(np.uint32))
        assert np.all(got[~nonzero] == 0)


@pytest.mark.parametrize("small", [False, True])
def test_binom_count(gpu, oracle, small):
    rng = np.random.default_rng(23)
    n = 1 << 21
    bits = rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32)
    bits[:64] = np.arange(64)
    bits[64:4096] = np.uint32(0xffffffff) - np.arange(4032, dtype=np.uint32)
    N = (rng.integers(2, 100, n) if small else np.rint(np.exp2(rng.uniform(np.log2(100), 24, n)))).astype(np.float32)
    x = np.where(rng.random(n) < 0.4, rng.random(n) * 12 / N, rng.random(n)).astype(np.float32)
    x = np.where(rng.random(n) < 0.3, np.float32(1) - x, x).astype(np.float32)
    x[::97], x[1::97] = 1.0, 0.0
    mean = (x * N).astype(np.float32)
    for k, edge in enumerate([np.float32(6), np.nextafter(np.float32(6), np.float32(7)), N[2::61] - np.float32(6), np.float32(np.nan)]):
        mean[2 + 15 * k::61] = edge if np.ndim(edge) == 0 else edge[:len(mean[2::61])]
    var = ((np.float32(1) - x) * mean).astype(np.float32)
    ok = ((mean >= 0) & (mean <= N)) | (mean != mean)
    bits, N, mean, var = bits[ok], N[ok], mean[ok], np.maximum(var[ok], np.float32(2.0 ** -96))
    got = gpu.device_math("binom_count", bits, mean, var, N)
    want = np.clip(oracle.binom_draw(bits, mean, var, N), 0, N.astype(np.int32))
    assert np.array_equal(got, want)
