"""The divisions of activation codes by way of a reciprocal (device_math.h: CodeDivisor, row_code_scale, quantize_code).
Their f32 steps are followed on the CPU over every mantissa; the kernels are held to the oracle's true divisions at the row
scales and next to the code boundaries where a reciprocal one unit off would show."""
import numpy as np
import pytest

F32, F64 = np.float32, np.float64


def _f32(a):
    """f32 values as doubles, which hold their products exactly."""
    return np.asarray(a, F32).astype(F64)


def _fma(a, b, c):
    """f32(a * b + c), rounded once.  The product of two f32 is exact in a double; the sum is rounded to odd there (its
    error, by Knuth's two-sum, decides the last bit), behind which a rounding to 24 bits is that of the exact sum."""
    p = np.multiply(a, b)
    s = p + c
    t = s - p
    err = (p - (s - t)) + (c - t)
    bits = s.view(np.int64)
    even = (bits & 1) == 0
    step = np.where((err > 0) == (s > 0), 1, -1)
    odd = np.where((err != 0) & even, bits + step, bits).view(F64)
    return odd.astype(F32).astype(F64)


def _mul(a, b):
    return np.multiply(a, b).astype(F32).astype(F64)


def _refined(s, start):
    """CodeDivisor's two Newton steps from a first reciprocal."""
    r = start
    for _ in range(2):
        r = _fma(_fma(-s, r, np.ones_like(s)), r, r)
    return r


def _divided(p, s, r):
    """div_by_uniform"""
    q = _mul(p, r)
    q = _fma(_fma(-q, s, p), r, q)
    return _fma(_fma(-q, s, p), r, q)


def _mantissas(first, last):
    return (np.arange(first, last, dtype=np.uint32) | np.uint32(0x3f800000)).view(F32)


def test_the_emulated_fma_is_rounded_once():
    from fractions import Fraction
    rng = np.random.default_rng(4)
    a, b = (_f32(rng.uniform(1, 2, 400)) for _ in range(2))
    c = _f32(-(a * b) * (1 + rng.choice([0.0, 2.0 ** -24, -2.0 ** -26, 0.3], 400)))
    for x, y, z, got in zip(a, b, c, _fma(a, b, c)):
        exact = Fraction(x) * Fraction(y) + Fraction(z)
        near = [F64(v) for v in (np.nextafter(F32(got), F32(-9)), F32(got), np.nextafter(F32(got), F32(9)))]
        best = min(abs(Fraction(v) - exact) for v in near)
        assert abs(Fraction(float(got)) - exact) == best


def test_reciprocals_of_every_mantissa():
    """From any start within two units in the last place (v_rcp_f32 is within one) the steps end at the correctly rounded
    reciprocal, of the largest mantissa at it or one unit below."""
    largest = set()
    for first in range(0, 1 << 23, 1 << 20):
        m = _mantissas(first, first + (1 << 20))
        s = _f32(m)
        right = (1.0 / s).astype(F32)  # (no quotient of 24-bit numbers is within 2^-53 of a rounding boundary)
        for off in range(-2, 3):
            start = _f32((right.view(np.int32) + off).view(F32))
            got = _refined(s, start).astype(F32).view(np.int32) - right.view(np.int32)
            if first + len(m) == 1 << 23:
                largest.add(int(got[-1]))
                got = got[:-1]
            assert (got == 0).all(), off
    assert largest <= {0, -1}


def test_scales_of_every_mantissa():
    """max / 127 with the constant of row_code_scale is the quotient of a true division."""
    recip, divisor = F64(F32(float.fromhex("0x1.020408p-7"))), F64(127.0)
    assert F32(recip) == F32(1.0) / F32(127.0)
    for first in range(0, 1 << 23, 1 << 20):
        m = _mantissas(first, first + (1 << 20))
        p = _f32(m)
        d = np.full_like(p, divisor)
        assert (_divided(p, d, np.full_like(p, recip)).astype(F32) == m / F32(127.0)).all()


# mantissas whose reciprocals are the hardest to round, and their neighbours
_EDGES = [0x7fffff, 0x7ffffe, 0x7ffffd, 0, 1, 2, 0x7f0000, 0x000100]


def _scale(mantissa, exponent):
    return np.array([(exponent + 127) << 23 | mantissa], np.uint32).view(F32)[0]


def _around_boundaries(s):
    """(n + 1/2) * s for every code boundary and up to four units in the last place beside it, both signs."""
    middle = ((np.arange(127) + 0.5) * F64(s)).astype(F32)
    x = (middle.view(np.int32)[:, None] + np.arange(-4, 5, dtype=np.int32)).view(F32).ravel()
    return np.concatenate([x, -x])


def test_the_largest_mantissa_needs_its_own_reciprocal():
    """One unit low, which the steps may leave it, the reciprocal gives other quotients, and codes: the correction of that
    one mantissa is needed, and it is enough.  Every other edge needs none."""
    for mantissa in _EDGES:
        s = F64(_scale(mantissa, 0))
        right = F64(F32(1.0 / s))
        x = _f32(_around_boundaries(s))
        want = (x.astype(F32) / F32(s)).astype(F64)
        sd = np.full_like(x, s)
        assert (_divided(x, sd, np.full_like(x, right)) == want).all(), hex(mantissa)
        if mantissa == 0x7fffff:
            low = F64(np.nextafter(F32(right), F32(0)))
            assert (np.rint(_divided(x, sd, np.full_like(x, low))) != np.rint(want)).any()


def _rows_with_scale(scales):
    """Rows whose largest element makes f32(max / 127) exactly the scale, the rest around its code boundaries."""
    rows = []
    for s in scales:
        top = F32(min(F64(s) * 127.0, 3.4e38))
        tops = (np.array([top], F32).view(np.int32) + np.arange(-2, 3, dtype=np.int32)).view(F32)
        tops = tops[np.isfinite(tops) & (tops / F32(127.0) == s)]
        if len(tops):
            body = np.clip(_around_boundaries(s), -tops[0], tops[0])
            rows.append(np.concatenate([[tops[0]], body, np.zeros(2304 - 1 - len(body), F32)]).astype(F32))
    return np.stack(rows)


_EXPONENTS = [-126, -125, -100, -62, -61, -60, -59, -1, 0, 1, 60, 100, 119, 120]


@pytest.mark.gpu
def test_codes_at_the_edges_of_the_reciprocal(ctx, oracle):
    import torch
    import volvoxai_amd.w8a8 as vx
    scales = [_scale(m, e) for m in _EDGES for e in _EXPONENTS]
    x = _rows_with_scale(scales)
    assert (x[:, 0] / F32(127.0)).view(np.uint32)[0] & 0x7fffff == 0x7fffff and len(x) > 60
    want, want_scales, finite = oracle.packed_prepare(x)
    assert finite.all()
    got, got_scales = vx.packed_prepare_i8(ctx, torch.from_numpy(x).cuda())
    assert (got_scales.cpu().numpy().view(np.uint32) == want_scales.view(np.uint32)).all()
    assert (got.cpu().numpy() == want).all()
    # the kernels that prepare one row and a few themselves: with unit scales one channel is the sum of the codes and the
    # next a weighted one, so that a code more or less shows
    k = x.shape[1]
    rng = np.random.default_rng(1)
    w = np.stack([np.ones(k, np.int8), rng.integers(-127, 128, k).astype(np.int8)])
    from volvoxai_amd.decoder import pack_w8_words
    words, sc = pack_w8_words(w), np.ones((2, k // 128), F32)
    pl = vx.PackedLinear(words, sc, None, k, 2, 128)
    for rows in (1, 2, 3):
        for first in range(0, len(x) - rows + 1, rows):
            if rows < 3 and first % (7 * rows):
                continue  # (a seventh of them)
            part = np.ascontiguousarray(x[first:first + rows])
            y_want = oracle.packed_linear(part, words, sc, None, 2, 128)[1]
            st, y = pl.forward_f32(ctx, torch.from_numpy(part).cuda())
            nan = np.isnan(y_want)  # (sums of the largest scales leave f32)
            y = y.cpu().numpy()
            assert st == 0 and (np.isnan(y) == nan).all() and (y.view(np.uint32) == y_want.view(np.uint32))[~nan].all(), (rows, first)
    pl.close()
    for s in scales:
        t = np.concatenate([_around_boundaries(s), np.array([np.inf, -np.inf, np.nan, 0.0, -0.0, 3e38, -3e38], F32)])
        for zp, dtype in ((0, vx.DTYPE_I8), (121, vx.DTYPE_U8)):
            ok, q = vx.quantize_typed_f32_i8u8(t, s, zp, dtype)
            assert ok == 1 and (q == oracle.quantize(t, s, zp, dtype)[1]).all(), (s, zp)


@pytest.mark.gpu
@pytest.mark.parametrize("exponent", [-120, -119, 0, 127])
def test_row_scales_of_every_mantissa(ctx, exponent):
    """Rows of one element: the scale is f32(max / 127), floored at 2^-126."""
    import torch
    import volvoxai_amd.w8a8 as vx
    for first in range(0, 1 << 23, 1 << 21):
        m = np.arange(first, first + (1 << 21), dtype=np.uint32) | np.uint32((exponent + 127) << 23)
        x = m.view(F32)[:, None]
        codes, scales = vx.packed_prepare_i8(ctx, torch.from_numpy(x).cuda())
        want = np.maximum(x[:, 0] / F32(127.0), F32(2.0 ** -126))
        assert (scales.cpu().numpy().view(np.uint32) == want.view(np.uint32)).all()
        assert (codes.cpu().numpy()[:, 0] == np.rint(np.minimum(x[:, 0] / want, F32(127.0)))).all()
