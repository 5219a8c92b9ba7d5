"""relu and the unary ops four elements a thread: bit for bit the one-element
kernels, which short and misaligned tensors take, on both sides of the line (2^18
elements), with remainders, zeros of both signs, infinities and NaN."""
import pytest
import torch

from pico_amd import kernels as K

pytestmark = pytest.mark.gpu

N0 = 1 << 18
OPS = ["sqrt", "sin", "cos", "tan", "tanh", "log", "relu"]


def _forward(op, x, y):
    return K.relu(x, y) if op == "relu" else K.unary(op, x, y)


def _backward(op, x, y, gy, gx, accumulate):
    if op == "relu":
        return K.relu_bwd(y, gy, gx, accumulate=accumulate)
    return K.unary_bwd(op, x, y, gy, gx, accumulate=accumulate)


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("n", [N0 - 1, N0, N0 + 1, N0 + 7, 5 * N0 + 2, 17 * N0 + 3])
@pytest.mark.parametrize("shift", [0, 1])
def test_wide_equals_narrow(dev, op, n, shift):
    g = torch.Generator(device=dev).manual_seed(n)
    buf = torch.randn(4, n + shift, device=dev, generator=g) * 3
    buf[:, 5::97] = 0.0
    buf[:, 6::97] = -0.0
    buf[0, 7::1001], buf[0, 8::1001], buf[0, 9::1001] = float("inf"), float("-inf"), float("nan")
    x, gy, g0 = (buf[i].clone()[shift:] for i in (0, 1, 2))
    y = torch.empty(n + shift, device=dev)[shift:]
    _forward(op, x, y)
    parts = [slice(i, min(i + N0 // 2, n)) for i in range(0, n, N0 // 2)]
    want = torch.empty(n, device=dev)
    for s in parts:
        _forward(op, x[s], want[s])
    assert torch.equal(y.view(torch.int32), want.view(torch.int32))
    for accumulate in (False, True):
        got, ref = g0.clone(), g0.clone()
        _backward(op, x, y, gy, got, accumulate)
        for s in parts:
            _backward(op, x[s], y[s], gy[s], ref[s], accumulate)
        assert torch.equal(got.view(torch.int32), ref.view(torch.int32))
