"""The bf16 and split-bf16 products of fp32 operands (gemm_narrow.hip) at the
edges of their tiles and slices.

Bounds against float64.  bf16: operands rounded to bf16 multiply exactly in
fp32, so only the sums round: a matrix instruction of 16 k at most 4 times,
each at most 2^-23 of the partial sums' bound sum |a||b| (the matrix unit may
truncate).  Split bf16: three such products per 16 k; rounding to bf16's 8
significant bits is off by 2^-8 at most, so hi leaves 2^-8 |x|, lo leaves
2^-16 |x| of that, once per operand, and lo.lo, at most 2^-16 |a||b|, is left
out: 3 2^-16 |a||b| together.
"""
import pytest
import torch

from pico_amd import kernels as K

pytestmark = pytest.mark.gpu

PRODUCT = {"bf16": K.gemm_bf16, "bf16x3": K.gemm_bf16x3}
LAYOUTS = [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")]


def _check(C, A, B, kind):
    Kd = A.shape[1]
    if kind == "bf16":
        a, b = A.bfloat16().double(), B.bfloat16().double()
        tol = (0.25 * Kd + 4) * 2.0 ** -23
    else:
        a, b = A.double(), B.double()
        tol = (0.75 * Kd + 4) * 2.0 ** -23 + 3 * 2.0 ** -16
    err = (C.double() - a @ b).abs()
    assert bool((err <= tol * (a.abs() @ b.abs())).all())


def _inside(x):
    """x as a strided view into a buffer of NaN, at an odd 4-byte offset"""
    buf = torch.full((x.shape[0] + 40, x.shape[1] + 3), float("nan"), device=x.device)
    buf[1:x.shape[0] + 1, 1:x.shape[1] + 1] = x
    return buf[1:x.shape[0] + 1, 1:x.shape[1] + 1]


# 256 x 256, 128 x 128, 256 x 96 and 64 x 64 tiles, whole and ragged; K of a part
# of a step, of a slice, whole slices odd and even in number; with a K split
@pytest.mark.parametrize("kind", ["bf16", "bf16x3"])
@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("M,N,Kd", [(4096, 4096, 64), (4095, 4097, 41), (2048, 2048, 96),
                                    (2047, 2049, 15), (8192, 768, 32), (8190, 768, 33),
                                    (1024, 1024, 160), (1023, 1021, 31), (515, 2047, 1),
                                    (5, 3, 127), (768, 768, 4096), (517, 301, 3001),
                                    # many slices inside the operands, then the bounded ones; rows
                                    # so short that a tile runs over several k rows
                                    (2049, 2047, 500), (8, 700, 303), (700, 6, 300), (200, 72, 97)])
def test_products_at_tile_edges(dev, kind, ta, tb, M, N, Kd):
    g = torch.Generator(device=dev).manual_seed(M + N + Kd)
    A = torch.randn(M, Kd, device=dev, generator=g)
    B = torch.randn(Kd, N, device=dev, generator=g)
    C = torch.full((M, N), float("nan"), device=dev)
    a, b = (A if ta == "N" else A.t()), (B if tb == "N" else B.t())
    whole = M % 32 == 0 and N % 32 == 0 and Kd % 32 == 0
    a, b = (a.contiguous(), b.contiguous()) if whole else (_inside(a), _inside(b))
    ws = torch.full((K.gemm_workspace(M, N, Kd) // 4,), float("nan"), device=dev)
    PRODUCT[kind](ta, tb, a, b, C, ws=ws if ws.numel() else None)
    _check(C, A, B, kind)


@pytest.mark.parametrize("kind", ["bf16", "bf16x3"])
@pytest.mark.parametrize("ta", ["N", "T"])
def test_rows_too_far_apart_for_buffer_offsets(dev, kind, ta):
    """a leading dimension above 2^21 (k-contiguous) or 2^24 floats: 64-bit
    addresses, the same result bit for bit as close rows give"""
    M, N, Kd = (3, 70, 1503) if ta == "N" else (67, 70, 35)
    ld = (1 << 21) + 8 if ta == "N" else (1 << 24) + 4
    g = torch.Generator(device=dev).manual_seed(7)
    A = torch.randn(M, Kd, device=dev, generator=g)
    B = torch.randn(Kd, N, device=dev, generator=g)
    a = (A if ta == "N" else A.t()).contiguous()
    far = torch.empty(a.shape[0], ld, device=dev)[:, :a.shape[1]]
    far.copy_(a)
    C, R = torch.empty(M, N, device=dev), torch.empty(M, N, device=dev)
    PRODUCT[kind](ta, "N", far, B, C)
    PRODUCT[kind](ta, "N", a, B, R)
    assert torch.equal(C, R)
    _check(C, A, B, kind)
