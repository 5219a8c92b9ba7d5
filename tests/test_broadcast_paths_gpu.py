"""The two-dimensional broadcast kernels and the ordered sums of a broadcast
operand's gradient, at the edges of their rules: bit for bit the oracle's (pico's
order and rounding), on both sides of each line, with odd sizes, signed zeros,
infinities and NaN among the terms."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from pico_amd import kernels as K

pytestmark = pytest.mark.gpu

# 31/32 terms and 8192/8193 columns are the lines of the ordered sums; 512/513 terms and
# 4096/4097 elements those of their long chunks; chunks hold 64, 256 or 1024 terms
SHAPES = [((31, 20), (20,)), ((32, 17), (17,)), ((65, 16), (16,)), ((513, 33), (33,)),
          ((1025, 4), (4,)), ((2049, 5), (5,)), ((40, 8192), (8192,)), ((40, 8193), (8193,)),
          ((600, 4097), (4097,)),
          ((20, 31), (20, 1)), ((17, 33), (17, 1)), ((5, 1030), (5, 1)), ((3, 2052), (3, 1)),
          ((8200, 40), (8200, 1)), ((4100, 513), (4100, 1)),
          # one row of more than 64 workgroups; rows either side of 70 % of their lanes
          ((500, 600), (1,)), ((90, 9), (9,)), ((90, 23), (90, 1)), ((90, 22), (22,)), ((9, 257), (9, 1)),
          ((37, 41), (1,)), ((1, 700), (1, 1)), ((6, 50, 7), (50, 7)), ((6, 50, 7), (6, 1, 1)),
          ((6, 50, 7), (50, 1)), ((4, 8, 64), (1, 8, 1)), ((3, 33, 2, 5), (33, 2, 1))]


def _values(shape, seed):
    a = O.normal(int(np.prod(shape)), seed).reshape(shape)
    f = a.ravel()
    f[::7] = -0.0
    f[::13] = 0.0
    return a


@pytest.mark.parametrize("op", [0, 1, 2])
@pytest.mark.parametrize("sa,sb", SHAPES)
def test_broadcast_bit_for_bit(dev, op, sa, sb):
    name = ["add", "sub", "mul"][op]
    a, b = _values(sa, 1), _values(sb, 2)

    def cu(x):
        return torch.from_numpy(np.ascontiguousarray(x)).to(dev)

    for x, y in ((a, b), (b, a)):
        out = K.binary(name, cu(x), cu(y))
        want = O.binary(op, x, y)
        assert np.array_equal(out.cpu().numpy().view(np.int32), want.view(np.int32))
    g = _values(sa, 3)
    for accumulate in (False, True):
        ga0, gb0 = (_values(s, 4) if accumulate else np.zeros(s, np.float32) for s in (sa, sb))
        for first in (True, False):  # the broadcast operand second, then first
            x, y, gx0, gy0 = (a, b, ga0, gb0) if first else (b, a, gb0, ga0)
            want = O.binary_bwd(op, x, y, g, gx0.copy(), gy0.copy())
            for which, s, so, other, g0, w in ((0, x.shape, y.shape, y, gx0, want[0]),
                                               (1, y.shape, x.shape, x, gy0, want[1])):
                got = cu(g0) if accumulate else torch.full(s, float("nan"), device=dev)
                K.binary_bwd(name, which, g.shape, s, so, cu(g), cu(other), got,
                             accumulate=accumulate)
                assert np.array_equal(got.cpu().numpy().view(np.int32), w.view(np.int32)), (which, s)


@pytest.mark.parametrize("R,C,axis", [(700, 40, 0), (40, 700, 1)])
def test_sums_of_infinities_and_nan(dev, R, C, axis):
    g = O.normal(R * C, 5).reshape(R, C)
    g[3, 5], g[20, 7], g[30, 7], g[10, 9] = np.inf, np.inf, -np.inf, np.nan
    shape = (C,) if axis == 0 else (R, 1)
    got = torch.empty(shape, device=dev)
    gd = torch.from_numpy(g).to(dev)
    K.binary_bwd("add", 1, (R, C), shape, (R, C), gd, gd, got)
    want = np.zeros(shape, np.float32)
    O.binary_bwd(0, g, np.zeros(shape, np.float32), g, np.zeros_like(g), want)
    assert np.array_equal(got.cpu().numpy(), want, equal_nan=True)
