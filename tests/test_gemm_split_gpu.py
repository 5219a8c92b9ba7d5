"""The fp32 product on the bf16 matrix cores (gemm_split.h): every operand is
the exact sum of three bf16 parts, six of whose nine products are added.

Bound of a sum over K terms: a matrix instruction of 16 k rounds its fp32
accumulator at most 4 times, six of them per 16 k, each rounding at most
2^-24 of the partial sums' bound sum |a||b|; the three products left out are
below 2^-24 of |a||b| together, and the K groups and the scaling add a few
more: |error| <= (1.5 K + 8) 2^-24 sum |a||b|.
"""
import numpy as np
import pytest
import torch

from pico_amd import kernels as K

pytestmark = pytest.mark.gpu


def _gen(seed):
    return torch.Generator(device="cuda:0").manual_seed(seed)


def _product(ta, tb, A, B, C, **kw):
    return K.gemm(ta, tb, A if ta == "N" else A.t().contiguous(),
                  B if tb == "N" else B.t().contiguous(), C, **kw)


def _within_bound(C, A, B):
    a, b = A.double(), B.double()
    err = (C.double() - a @ b).abs()
    return bool((err <= (1.5 * A.shape[1] + 8) * 2.0 ** -24 * (a.abs() @ b.abs())).all())


# whole and ragged sizes of every tile: 256 x 256, 128 x 128, 256 x 96, 64 x 64; K of a
# part of a slice, one slice, an odd number of slices, and past a sign change of the sums
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("M,N,Kd", [(4096, 4096, 64), (4096, 4099, 200), (2048, 2048, 32),
                                    (2047, 1985, 17), (8192, 768, 64), (8191, 768, 130),
                                    (4096, 768, 64), (4095, 768, 49), (1024, 1024, 128),
                                    (1023, 1021, 131), (515, 2047, 1), (700, 600, 1100),
                                    # 64 x 64 tiles with one and two wave groups
                                    (1184, 448, 32), (601, 930, 10), (1103, 577, 48), (1472, 192, 192),
                                    (1024, 1024, 256), (601, 930, 200), (601, 930, 257)])
def test_within_fp32_bound(dev, ta, tb, M, N, Kd):
    g = _gen(M + N + Kd)
    A = torch.randn(M, Kd, device=dev, generator=g)
    B = torch.rand(Kd, N, device=dev, generator=g)
    C = torch.full((M, N), float("nan"), device=dev)
    _product(ta, tb, A, B, C)
    assert _within_bound(C, A, B)


# 256 x 256, 128 x 128, 256 x 96, 64 x 64 and 128 x 64 tiles, and a K split
@pytest.mark.parametrize("ta,M,N,Kd", [("N", 4096, 4096, 768), ("N", 4096, 4096, 2048), ("N", 2048, 2048, 2048),
                                       ("N", 8192, 768, 768), ("N", 1100, 1100, 1024), ("N", 1100, 1100, 200),
                                       ("N", 4096, 512, 512), ("T", 512, 512, 4096)])
def test_errors_do_not_share_a_sign(dev, ta, M, N, Kd):
    """the matrix unit drops bits of small products towards minus infinity; the
    alternating sign of the sums keeps that out of the result.  The mean error
    over M N outputs is within 8 standard errors of independent ones, plus what
    256 x 256 tiles leave of the last 128 k between two turns (1.3 of K / rms measured
    from K 256 on, the bound allows 3); the means of columns, of M outputs
    each, spread as independent errors do, and twice that at most"""
    g = _gen(5)
    A = torch.randn(M, Kd, device=dev, generator=g)
    B = torch.randn(Kd, N, device=dev, generator=g)
    C = torch.empty(M, N, device=dev)
    ws = torch.full((K.gemm_workspace(M, N, Kd) // 4 + 4,), float("nan"), device=dev)
    K.gemm_ex(ta, "N", A if ta == "N" else A.t().contiguous(), B, C, ws=ws)
    e = C.double() - A.double() @ B.double()
    rms = float(e.square().mean().sqrt())
    turns = 3 / Kd if M * N >= 4096 * 4096 else 0
    assert abs(float(e.mean())) <= (8 / (M * N) ** 0.5 + turns) * rms
    assert float(e.mean(0).square().mean().sqrt()) <= 2 * rms / M ** 0.5


# relative 2-norm error of the fp32 matrix instructions these products replaced
# (one rounding a k), measured with the kernel that ran before on [2048, 2048]
FP32_CORES = {16: {"normal": 7.37e-8, "unit": 6.20e-8, "relu": 5.51e-8, "prob": 6.92e-8},
              64: {"normal": 1.45e-7, "unit": 1.15e-7, "relu": 1.04e-7, "prob": 1.31e-7},
              512: {"normal": 4.06e-7, "unit": 3.06e-7, "relu": 2.85e-7, "prob": 3.58e-7},
              2048: {"normal": 8.11e-7, "unit": 6.00e-7, "relu": 5.72e-7, "prob": 7.75e-7}}


@pytest.mark.parametrize("M,N", [(4096, 4096), (2048, 2048), (8192, 768), (1100, 1100)])
@pytest.mark.parametrize("Kd", [16, 64, 512, 2048])
@pytest.mark.parametrize("kind", ["normal", "unit", "relu", "prob"])
def test_error_against_the_fp32_cores(dev, M, N, Kd, kind):
    """operands of both signs, of one sign (uniform in [0, 1), probabilities
    times values around 1) and half zeros: no more error than fp32 multiplies
    had (1 % for the sample), but for half zeros in 256 x 256 tiles, measured
    1.03 (K 64) to 1.15 times theirs"""
    g = _gen(Kd + M)
    A = torch.randn(M, Kd, device=dev, generator=g)
    B = torch.randn(Kd, N, device=dev, generator=g)
    if kind == "unit":
        A, B = torch.rand(M, Kd, device=dev, generator=g), torch.rand(Kd, N, device=dev, generator=g)
    elif kind == "relu":
        A = A.relu()
    elif kind == "prob":
        A, B = (3 * A).softmax(1), B + 1
    C = torch.empty(M, N, device=dev)
    K.gemm("N", "N", A, B, C)
    R = A.double() @ B.double()
    err = float((C.double() - R).norm() / R.norm())
    largest = kind == "relu" and M == 4096 and Kd >= 64
    assert err <= (1.17 if largest else 1.01) * FP32_CORES[Kd][kind]


# K split with a partial last slice, odd leading dimensions at odd 4-byte offsets, and
# a workspace and surroundings of NaN: 64 x 64 (130x70, 517x301) and 128-row tiles,
# and whole 128 x 64 ones
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("M,N,Kd", [(517, 301, 3001), (130, 70, 5001), (768, 768, 8191), (512, 512, 4096)])
@pytest.mark.parametrize("bad", [False, True])
def test_k_split(dev, ta, tb, M, N, Kd, bad):
    g = _gen(M + Kd)
    A = torch.randn(M, Kd, device=dev, generator=g)
    B = torch.randn(Kd, N, device=dev, generator=g)
    if bad:  # inside one split, and in the last, partial slice
        A[5, Kd // 2], B[Kd - 1, 7] = float("inf"), float("nan")

    def inside(x):
        buf = torch.full((x.shape[0] + 40, x.shape[1] + 3), float("nan"), device=dev)
        buf[1:x.shape[0] + 1, 1:x.shape[1] + 1] = x
        return buf[1:x.shape[0] + 1, 1:x.shape[1] + 1]

    need = K.gemm_workspace(M, N, Kd)
    assert need > 0
    ws = torch.full((need // 4,), float("nan"), device=dev)
    X = torch.randn(M, N, device=dev, generator=g)
    C = X.clone()
    K.gemm_ex(ta, tb, inside(A if ta == "N" else A.t()), inside(B if tb == "N" else B.t()), C, beta=0.5, ws=ws)
    if bad:
        assert bool(torch.isnan(C[:, 7]).all())
        rest = torch.cat([C[5, :7], C[5, 8:]])
        sign = torch.cat([B[Kd // 2, :7], B[Kd // 2, 8:]]).sign()
        assert torch.equal(rest, sign * float("inf"))
        A[5], B[:, 7], C[5], C[:, 7], X[5], X[:, 7] = 0.0, 0.0, 0.0, 0.0, 0.0, 0.0
    a, b = A.double(), B.double()
    err = (C.double() - 0.5 * X.double() - a @ b).abs()
    assert bool((err <= (1.5 * Kd + 80) * 2.0 ** -24 * (a.abs() @ b.abs() + X.double().abs())).all())


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("T", "N")])
def test_every_float_passes_exactly(dev, ta, tb):
    """times the identity, any finite float (subnormal and near the largest
    among them) comes back bit for bit: the three parts hold all 24 bits, and
    what overflows the scaled sums is computed again on the fp32 cores"""
    bits = torch.randint(0, 1 << 32, (600, 1040), generator=_gen(1), device=dev, dtype=torch.int64)
    A = (bits - (1 << 31)).to(torch.int32).view(torch.float32)
    A = torch.where(torch.isfinite(A), A, torch.ones_like(A))
    one = torch.eye(1040, device=dev)
    for rows in (A, torch.ldexp(A.sign(), torch.randint(-149, 128, A.shape, generator=_gen(2),
                                                        device=dev).float())):
        # one magnitude per row and group of columns, so the sums are single values
        C = torch.empty(600, 1040, device=dev)
        _product(ta, tb, rows, one, C)
        assert torch.equal(C, rows + 0.0)


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N")])
def test_infinities_and_nan(dev, ta, tb):
    M, N, Kd = 1100, 700, 1500
    g = _gen(3)
    A = torch.randn(M, Kd, device=dev, generator=g)
    B = torch.randn(Kd, N, device=dev, generator=g)
    A[3, 7], A[500, 1499], A[1099, 0] = float("inf"), float("nan"), float("-inf")
    A[200, 5] = 3e38  # rounds to an infinite bf16
    B[7, 11] = 0.0
    C = torch.empty(M, N, device=dev)
    _product(ta, tb, A, B, C)
    R = A.double() @ B.double()
    assert torch.equal(torch.isnan(C), torch.isnan(R))
    assert bool(torch.isnan(C[500]).all()) and bool(torch.isnan(C[3, 11]))
    inf = torch.isinf(R) | (R.abs() > 3.4028235e38)
    assert torch.equal(C[inf].double().sign(), R[inf].sign()) and bool(torch.isinf(C[inf]).all())
    fine = torch.ones(M, dtype=torch.bool, device=dev)
    fine[[3, 200, 500, 1099]] = False
    assert _within_bound(C[fine], A[fine], B)


@pytest.mark.parametrize("ta,tb,M,N,Kd", [("N", "N", 3, 5, 1500), ("N", "T", 70, 130, 1503),
                                          ("N", "N", 128, 64, 4096), ("T", "N", 67, 70, 35)])
def test_rows_too_far_apart_for_buffer_offsets(dev, ta, tb, M, N, Kd):
    """a leading dimension above 2^21 (k-contiguous) or 2^25 floats: 64-bit
    addresses, also with K split and a residual"""
    ld = (1 << 21) + 8 if ta == "N" else (1 << 25) + 4
    A = torch.randn(M, Kd, device=dev, generator=_gen(4))
    B = torch.randn(Kd, N, device=dev, generator=_gen(5))
    a = A if ta == "N" else A.t()
    far = torch.full((a.shape[0], ld), float("nan"), device=dev)[:, :a.shape[1]]
    far.copy_(a)
    b = B if tb == "N" else B.t().contiguous()
    for ws in (None, torch.full((K.gemm_workspace(M, N, Kd) // 4 + 4,), float("nan"), device=dev)):
        C = torch.full((M, N), 3.0, device=dev)
        if ws is None:
            K.gemm(ta, tb, far, b, C)
        else:
            K.gemm_ex(ta, tb, far, b, C, beta=1.0, ws=ws)
            C = C.double() - 3.0
        a64, b64 = A.double(), B.double()
        err = (C.double() - a64 @ b64).abs()
        assert bool((err <= (1.5 * Kd + 10) * 2.0 ** -24 * (a64.abs() @ b64.abs() + 3.0)).all())


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("T", "N"), ("N", "T")])
def test_ragged_operands_end_where_they_end(dev, ta, tb):
    """strided, ragged operands inside buffers of NaN: nothing outside them
    reaches the result"""
    M, N, Kd = 517, 1031, 1203
    g = _gen(6)
    A = torch.randn(M, Kd, device=dev, generator=g)
    B = torch.randn(Kd, N, device=dev, generator=g)

    def inside(x):
        buf = torch.full((x.shape[0] + 64, x.shape[1] + 3), float("nan"), device=dev)
        buf[:x.shape[0], :x.shape[1]] = x
        return buf[:x.shape[0], :x.shape[1]]

    C = torch.full((M, N), float("nan"), device=dev)
    K.gemm(ta, tb, inside(A if ta == "N" else A.t()), inside(B if tb == "N" else B.t()), C)
    assert np.isfinite(C.cpu().numpy()).all() and _within_bound(C, A, B)


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("T", "N"), ("N", "T"), ("T", "T")])
@pytest.mark.parametrize("M,N,Kd", [(517, 1031, 1203), (4000, 4100, 100), (1100, 700, 70)])
def test_what_lies_behind_rows_does_not_choose_the_route(dev, ta, tb, M, N, Kd):
    """a tile's rows and columns past M and N may read what lies between an
    operand's rows: NaN there gives the same bits as zeros do, so no block
    was computed again for it"""
    g = _gen(8)
    A = torch.randn(M, Kd, device=dev, generator=g)
    B = torch.randn(Kd, N, device=dev, generator=g)

    def product(fill):
        def inside(x):
            buf = torch.full((x.shape[0] + 64, x.shape[1] + 300), fill, device=dev)
            buf[:x.shape[0], :x.shape[1]] = x
            return buf[:x.shape[0], :x.shape[1]]
        C = torch.full((M, N), 1.0, device=dev)
        K.gemm(ta, tb, inside(A if ta == "N" else A.t()), inside(B if tb == "N" else B.t()), C, beta=1.0)
        return C

    assert torch.equal(product(float("nan")), product(0.0))


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("M,N,Kd", [(4096, 4096, 77), (2048, 2048, 512), (1024, 1024, 33), (601, 930, 300),
                                    (4096, 512, 100), (8192, 768, 96)])
def test_one_row_and_column_not_finite(dev, ta, tb, M, N, Kd):
    """the other rows and columns keep their accuracy, beta's matrix is added once"""
    g = _gen(9)
    A = torch.randn(M, Kd, device=dev, generator=g)
    B = torch.randn(Kd, N, device=dev, generator=g)
    A[M // 3, Kd - 1], B[Kd // 2, N - 2] = float("inf"), float("nan")
    C = torch.full((M, N), 2.0, device=dev)
    _product(ta, tb, A, B, C, beta=1.0)
    assert bool(torch.isnan(C[:, N - 2]).all())
    rest = [i for i in range(N) if i != N - 2]
    row = C[M // 3][rest].double()
    assert bool((row == A[M // 3, Kd - 1].double() * B[Kd - 1][rest].double().sign()).all())
    A[M // 3], B[:, N - 2], C[M // 3], C[:, N - 2] = 0.0, 0.0, 2.0, 2.0
    a, b = A.double(), B.double()
    err = (C.double() - 2.0 - a @ b).abs()
    assert bool((err <= (1.5 * Kd + 10) * 2.0 ** -24 * (a.abs() @ b.abs() + 2.0)).all())


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("M,N", [(4096, 4096), (2047, 2049), (1100, 1100), (8192, 768)])
def test_single_products_are_rounded_once(dev, ta, tb, M, N):
    """K 1: every output is one fp32 product, correctly rounded; K 2: off by two
    roundings at most"""
    g = _gen(10)
    A = torch.randn(M, 2, device=dev, generator=g)
    B = torch.randn(2, N, device=dev, generator=g)
    C = torch.empty(M, N, device=dev)
    _product(ta, tb, A[:, :1].contiguous(), B[:1].contiguous(), C)
    assert torch.equal(C, A[:, :1] * B[:1])
    _product(ta, tb, A, B, C)
    a, b = A.double(), B.double()
    assert bool(((C.double() - a @ b).abs() <= 2 * 2.0 ** -24 * (a.abs() @ b.abs())).all())
