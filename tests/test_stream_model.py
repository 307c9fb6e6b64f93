"""CPU checks of the streamed kernels' arithmetic and LDS layout
(csrc/fused_stream_impl.h), restated here: three bf16 thirds carry a Float32
value exactly, the six partial products that the kernels form miss a product by
2^-23 of it at most and 2^-26 as a rule, and with the slot and column strides that the kernels use
every LDS read of a block falls on distinct banks."""
import numpy as np
import pytest


def bf16(x):
    """Round to nearest even, as a Float32 value."""
    u = x.view(np.uint32).astype(np.uint64)
    return (((u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000).astype(np.uint32)).view(np.float32)


def thirds(x):
    a = bf16(x)
    r = x - a
    b = (r.view(np.uint32) & np.uint32(0xffff0000)).view(np.float32)
    return a, b, r - b


def values(seed, n=200000):
    rng = np.random.default_rng(seed)
    return (rng.uniform(1, 2, n) * 2.0 ** rng.integers(-60, 60, n) * rng.choice([-1, 1], n)).astype(np.float32)


def test_thirds_are_exact():
    x = values(1)
    a, b, c = thirds(x)
    for t in (a, b, c):
        assert not (t.view(np.uint32) & 0xffff).any()  # bf16 values
    assert (a.astype(np.float64) + b + c == x).all()


def test_six_products():
    x, y = values(2), values(3)
    (a, b, c), (d, e, f) = ([t.astype(np.float64) for t in thirds(z)] for z in (x, y))
    got = c * d + a * f + b * e + b * d + a * e + a * d
    err = (got - x.astype(np.float64) * y) / np.abs(x.astype(np.float64) * y)
    assert np.abs(err).max() < 2.0 ** -23 and np.sqrt((err ** 2).mean()) < 2.0 ** -26
    assert abs(err.mean()) < 2.0 ** -32  # (of either sign)


def test_halves_lose_small_components():
    """What two f16 halves under one scale (the largest value in [4, 8)) would keep."""
    big, small = np.float32(1.0), np.float32(1.2345e-6)
    s = np.float32(4.0 / big)
    hi = np.float16(small * s)
    lo = np.float16(small * s - np.float32(hi))
    assert abs((float(hi) + float(lo)) / float(s) / float(small) - 1) > 1e-3
    assert sum(float(t[0]) for t in thirds(np.array([small]))) == float(small)


B128 = [[0, 1, 2, 3, 12, 13, 14, 15, 20, 21, 22, 23, 24, 25, 26, 27],
        [4, 5, 6, 7, 8, 9, 10, 11, 16, 17, 18, 19, 28, 29, 30, 31]]


@pytest.mark.parametrize("NT", [1, 2, 3, 4])
@pytest.mark.parametrize("one", [False, True])
@pytest.mark.parametrize("hr", [16, 20, 24, 36, 48, 60])
def test_block_reads_conflict_free(NT, one, hr):
    SB = 192 * NT + 32
    cr = hr + ((4 - hr % 8) + 8) % 8

    def slot(e):  # element e of a block
        return e if one else (e & 3) + cr * (e >> 2)
    for group in B128 + [[i + 32 for i in g] for g in B128]:  # 16-byte rows: lane j + 16 g
        for third in (False, True):  # ([c | a] of an odd last group)
            units = set()
            for i in group:
                j, g = i & 15, i >> 4
                off = 16 * g + ((64 if g < 2 else -32) if third else 0)
                units.add((slot(j) * SB + off) // 16 % 16)
            assert len(units) == 16
    for half in range(2):  # transposing reads: 8 bytes a lane, 32 lanes
        banks = set()
        for i in range(32 * half, 32 * half + 32):
            j, g = i & 15, i >> 4
            a = slot(4 * g + (j >> 2)) * SB + 8 * (j & 3)
            banks |= {a // 4 % 64, a // 4 % 64 + 1}
        assert len(banks) == 64
