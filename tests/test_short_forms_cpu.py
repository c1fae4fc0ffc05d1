"""The short reciprocal and quotient of the kernels (bnx_numeric.h, compiled for
the host): against the division over all mantissas and on quotients next to a
midpoint, and where their callers have to look at a range.  A cell of the march
next to an alpha of 0 in the transfer function has a majorant as small as its
scalars, down to the smallest subnormal: the quotient by it has to be the
division's there too, and a draw has to leave the cell.  A cell inversion's
determinant may be as large as floats get.

Reciprocal estimates are as far off as the hardware's, less than an ulp: the
rounded reciprocal, or (far) the float on the other side of the exact one; for
a mantissa of ones, where a step from the latter does not reach the former, the
hardware's is the former."""
import numpy as np

from barney_amd import abi


ONES = np.float32(2 - 2.0 ** -23)


def test_reciprocal_of_every_mantissa(orc):
    b = (np.arange(1 << 23, dtype=np.uint32) | np.uint32(127 << 23)).view(np.float32)
    for far in (0, 1):
        out = np.empty_like(b)
        orc.lib().orc_rcp_n(abi.fptr(b), far, len(b), abi.fptr(out))
        bad = b[out != np.float32(1) / b]
        assert len(bad) == 0 or (far == 1 and list(bad) == [ONES]), (far, bad[:5])


def _quotient(orc, a, b, far=0, scale=1.0):
    a, b = (np.ascontiguousarray(x, np.float32) for x in np.broadcast_arrays(a, b))
    out = np.empty_like(a)
    orc.lib().orc_div_n(abi.fptr(a), abi.fptr(b), scale, far, a.size, abi.fptr(out))
    return out


def test_quotients_next_to_midpoints(orc):
    """a / b = q + half an ulp, nearly: for an odd m = 2q + 1 (25 bits) and an odd b, the a with 2^25 a = m b -+ r for
    the smallest remainders r.  Solved modulo 2^k for many b, and checked in integers."""
    r = np.random.default_rng(3)
    a_all, b_all = [], []
    bits = 25
    for b in list(range((1 << 24) - 199, 1 << 24, 2)) + [int(x) | 1 for x in r.integers(1 << 23, 1 << 24, 3000)]:
        inv = pow(b, -1, 1 << bits)
        for rem in (-5, -3, -1, 1, 3, 5):
            m = (rem * inv) % (1 << bits)                 # m b = rem (mod 2^25)
            if m & 1 and (1 << 24) <= m < (1 << 25):
                a = (m * b - rem) >> bits
                if (1 << 23) <= a < (1 << 24) or (1 << 22) <= a < (1 << 23):
                    a_all.append(a)
                    b_all.append(b)
    a, b = np.array(a_all, np.float32), np.array(b_all, np.float32)
    assert len(a) > 3000 and (a.astype(np.int64) == a_all).all()
    want = a / b
    for far in (0, 1):
        ok = b != np.float32((1 << 24) - 1)
        for e in (-60, 0, 75):
            s = np.float32(2.0 ** e)
            assert np.array_equal(_quotient(orc, a[ok], b[ok] * s, far), want[ok] / s)


def test_quotients_by_determinants(orc):
    scale = orc.lib().orc_det_scale()
    d = _majorants(-60, 128)
    d = np.concatenate([d, -d])
    ok = np.abs(np.frexp(d)[0]) != ONES / 2
    for part in (1.0, 0.5, -0.37, 1e-3, 1e-6, 1e-12, 0.0):
        a = (d * np.float32(part)).astype(np.float32)
        assert np.array_equal(_quotient(orc, a, d, scale=scale), a / d)
        assert np.array_equal(_quotient(orc, a[ok], d[ok], 1, scale), a[ok] / d[ok])
    # what the scale is for: a step of 0 where it is half the cell
    top = _majorants(127, 128)
    assert (_quotient(orc, top / 2, top) == 0).all()


def _over(orc, x, maj, far, guard=1):
    x, maj = (np.ascontiguousarray(a, np.float32) for a in np.broadcast_arrays(x, maj))
    out = np.empty(x.size, np.float32)
    orc.lib().orc_over_majorant_n(abi.fptr(x.reshape(-1)), abi.fptr(maj.reshape(-1)), far, guard, x.size,
                                  abi.fptr(out))
    return out.reshape(x.shape)


def _majorants(lo, hi, n=400, ones=True):
    """n a binade of [2^lo, 2^hi), its ends among them"""
    r = np.random.default_rng(1)
    m = np.concatenate([[1.0, 1 + 2.0 ** -23, 2 - 2.0 ** -(22 + ones)], r.uniform(1, 2 - 2.0 ** -21, n)])
    e = np.arange(lo, hi)[:, None]
    return np.unique((m * 2.0 ** e).astype(np.float32).reshape(-1))


def _steps():
    """the free path's numerators, -log(1 - draw): 0 and 2^-24 to 3.1"""
    r = np.random.default_rng(2)
    return np.concatenate([[0.0, 2.0 ** -24, 2.0 ** -23, 0.5, 3.0666666], r.uniform(0, 3.07, 40)]).astype(np.float32)


def test_quotient_by_any_majorant(orc):
    with np.errstate(over="ignore"):
        for far in (0, 1):
            maj = _majorants(-149, 50, ones=far == 0)
            assert maj[0] == np.float32(2.0 ** -149)
            for x in _steps():
                assert np.array_equal(_over(orc, x, maj, far), np.float32(x) / maj), (x, far)
            # a density over the majorant, the ratio that a shadow ray's estimate takes
            for part in (1.0, 0.999, 0.37, 2.0 ** -10):
                s = (maj * np.float32(part)).astype(np.float32)
                assert np.array_equal(_over(orc, s, maj, far), s / maj), (part, far)


def test_draws_leave_cells_of_tiny_majorants(orc):
    maj = _majorants(-149, -100)
    for x in _steps()[1:]:
        t = np.float32(0.25) + _over(orc, x, maj, 0)
        assert (t >= np.float32(1.75)).all()
    # what the look at the majorant is for: without it the path has no length
    assert np.isnan(_over(orc, 0.5, _majorants(-149, -129), 0, guard=0)).all()
