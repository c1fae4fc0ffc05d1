"""The march's short quotient by a macrocell's majorant (bnx_numeric.h, compiled
for the host), with reciprocal estimates as far off as the hardware's (v_rcp_f32:
within 1 ulp, and the rounded reciprocal itself for a mantissa of ones, the one
that a step from the ulp beside it does not mend): a cell next to an alpha of 0 in the transfer function has a
majorant as small as its scalars, down to the smallest subnormal.  The quotient
has to be the division's there too, and a draw has to leave the cell."""
import numpy as np

from barney_amd import abi


def _over(orc, x, maj, ulps, guard=1):
    x, maj = (np.ascontiguousarray(a, np.float32) for a in np.broadcast_arrays(x, maj))
    out = np.empty(x.size, np.float32)
    orc.lib().orc_over_majorant_n(abi.fptr(x.reshape(-1)), abi.fptr(maj.reshape(-1)), ulps, guard, x.size,
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
        for ulps in (-1, 0, 1):
            maj = _majorants(-149, 50, ones=ulps == 0)
            assert maj[0] == np.float32(2.0 ** -149)
            for x in _steps():
                assert np.array_equal(_over(orc, x, maj, ulps), np.float32(x) / maj), (x, ulps)
            # a density over the majorant, the ratio that a shadow ray's estimate takes
            for part in (1.0, 0.999, 0.37, 2.0 ** -10):
                s = (maj * np.float32(part)).astype(np.float32)
                assert np.array_equal(_over(orc, s, maj, ulps), s / maj), (part, ulps)


def test_draws_leave_cells_of_tiny_majorants(orc):
    maj = _majorants(-149, -100)
    for x in _steps()[1:]:
        t = np.float32(0.25) + _over(orc, x, maj, 0)
        assert (t >= np.float32(1.75)).all()
    # what the look at the majorant is for: without it the path has no length
    assert np.isnan(_over(orc, 0.5, _majorants(-149, -129), 0, guard=0)).all()
