"""Fused attention of head sizes 32, 96 and 128 (pk_flash_wide_*) against float64,
at the edges of its 32-row blocks and of its 64- and 128-row workgroups.

Bound: every output is a sum of at most T terms, and every term a product whose
factors come from sums of hd terms, all in fp32: relative error (2-norm) below
(hd + T) 2^-24 at worst and about its square root in fact; 1e-5 covers T 1040."""
import ctypes

import numpy as np
import pytest
import torch

from pico_amd import _lib
from pico_amd.pico import Pico

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _fwd(B, H, T, hd, ld, q, k, v):
    o = torch.full((B * T, H * hd), float("nan"), device=q.device)
    lse = torch.full((B * H * T,), float("nan"), device=q.device)
    st = torch.cuda.current_stream().cuda_stream
    _lib.check("fwd", _lib.hip_lib().pk_flash_wide_fwd_f32(
        B, H, T, hd, ld, hd ** -0.5, _ptr(q), _ptr(k), _ptr(v), _ptr(o), _ptr(lse), st))
    return o, lse


def _bwd(B, H, T, hd, ld, q, k, v, o, lse, do, grads, flags=0):
    L = _lib.hip_lib()
    need = L.pk_flash_wide_bwd_workspace(B, H, T)
    ws = torch.full((need // 4,), float("nan"), device=q.device)
    st = torch.cuda.current_stream().cuda_stream
    _lib.check("bwd", L.pk_flash_wide_bwd_f32(
        B, H, T, hd, ld, hd ** -0.5, _ptr(q), _ptr(k), _ptr(v), _ptr(o), _ptr(lse), _ptr(do),
        *(_ptr(g) for g in grads), _ptr(ws), need, flags, st))


def _reference(B, H, T, hd, q, k, v, do):
    x = [t.double().reshape(B, T, H, hd).transpose(1, 2).reshape(B * H, T, hd).contiguous()
         .requires_grad_() for t in (q, k, v)]
    s = torch.bmm(x[0], x[1].transpose(1, 2).contiguous()) * hd ** -0.5
    s = s.masked_fill(~torch.ones(T, T, dtype=torch.bool, device=q.device).tril(), float("-inf"))
    o = torch.bmm(torch.softmax(s, -1), x[2])

    def flat(t):
        return t.reshape(B, H, T, hd).transpose(1, 2).reshape(B * T, H * hd)

    flat(o).backward(do.double())
    return flat(o).detach(), torch.logsumexp(s, -1).reshape(-1).detach(), [flat(t.grad) for t in x]


def _close(got, want):
    err = float((got.double() - want).norm() / want.norm().clamp_min(1e-30))
    assert np.isfinite(err) and err <= TOL, err


# two-wave workgroups, then four-wave ones (at least 512 blocks of 128 rows)
@pytest.mark.parametrize("hd", [32, 96, 128])
@pytest.mark.parametrize("B,H,T", [(1, 1, 1), (2, 3, 31), (1, 2, 32), (2, 1, 33), (1, 2, 64),
                                   (1, 3, 65), (2, 2, 100), (1, 2, 129), (1, 1, 1040),
                                   (16, 16, 130), (32, 16, 97)])
def test_against_float64(dev, hd, B, H, T):
    g = torch.Generator(device=dev).manual_seed(B * 1000 + T + hd)
    D = H * hd
    q, k, v, do = (torch.randn(B * T, D, device=dev, generator=g) for _ in range(4))
    o, lse = _fwd(B, H, T, hd, D, q, k, v)
    ro, rl, rg = _reference(B, H, T, hd, q, k, v, do)
    _close(o, ro)
    _close(lse, rl)
    grads = [torch.full_like(q, float("nan")) for _ in range(3)]
    _bwd(B, H, T, hd, D, q, k, v, o, lse, do, grads)
    for got, want in zip(grads, rg):
        if T > 1:
            _close(got, want)
        else:  # one key: the scores' gradient is exactly zero
            assert float((got.double() - want).abs().max()) <= 1e-5 * float(do.abs().max())


@pytest.mark.parametrize("hd", [32, 96, 128])
def test_column_views_accumulate_and_read_nothing_past_the_end(dev, hd):
    """q, k, v and their gradients as column blocks of one [B*T, 3*H*hd] matrix whose
    further rows are NaN; each flags bit adds onto its gradient"""
    B, H, T = 2, 2, 77
    D, g = H * hd, torch.Generator(device=dev).manual_seed(hd)
    buf = torch.full((B * T + 130, 3 * D), float("nan"), device=dev)
    buf[:B * T] = torch.randn(B * T, 3 * D, device=dev, generator=g)
    q, k, v = (buf[:B * T, i * D:(i + 1) * D] for i in range(3))
    do = torch.full((B * T + 130, D), float("nan"), device=dev)
    do[:B * T] = torch.randn(B * T, D, device=dev, generator=g)
    do = do[:B * T]
    o, lse = _fwd(B, H, T, hd, 3 * D, q, k, v)
    ro, _, rg = _reference(B, H, T, hd, q, k, v, do)
    _close(o, ro)
    for flags in range(8):
        grad = torch.full((B * T, 3 * D), 0.5, device=dev)
        views = [grad[:, i * D:(i + 1) * D] for i in range(3)]
        _bwd(B, H, T, hd, 3 * D, q, k, v, o, lse, do, views, flags)
        for i, want in enumerate(rg):
            _close(views[i], want + (0.5 if flags >> i & 1 else 0.0))


@pytest.mark.parametrize("hd", [96, 128])
@pytest.mark.parametrize("trend", ["rising", "falling"])
def test_running_max(dev, hd, trend):
    """keys whose scale grows along the sequence raise the running max on most
    blocks; shrinking ones leave the first block dominant"""
    B, H, T = 1, 2, 300
    g = torch.Generator(device=dev).manual_seed(9)
    q, k, v, do = (torch.randn(B * T, H * hd, device=dev, generator=g) for _ in range(4))
    ramp = torch.linspace(0.05, 8.0, T, device=dev)
    k = k * (ramp if trend == "rising" else ramp.flip(0))[:, None]
    o, lse = _fwd(B, H, T, hd, H * hd, q, k, v)
    ro, rl, _ = _reference(B, H, T, hd, q, k, v, do)
    _close(o, ro)
    _close(lse, rl)


def test_one_tensor_as_q_k_and_v_and_the_chain_beyond_the_cap(dev, monkeypatch):
    """attention(x, x, x) through pico: the three gradients add up in x's; with no
    room for the dS tiles the chain runs, within rounding of the same values"""
    P = Pico()
    B, H, T, hd = 2, 2, 70, 96
    x0 = np.random.default_rng(3).standard_normal((B * T, H * hd)).astype(np.float32)
    out = {}
    for cap in ("", "0"):
        monkeypatch.setenv("PICO_ATTN_DS_CAP", cap)
        with P.arena(1 << 26):
            x = P.param([B * T, H * hd], x0)
            y = P.attention_causal(x, x, x, B, H)
            P.backward(y)
            out[cap] = (P.data(y), P.grad(x))
            P.free(x)
    q = torch.from_numpy(x0).to(dev)
    ro, _, rg = _reference(B, H, T, hd, q, q, q, torch.ones_like(q))
    for y, dx in out.values():
        _close(torch.from_numpy(y).to(dev).reshape(ro.shape), ro)
        _close(torch.from_numpy(dx).to(dev).reshape(ro.shape), sum(rg))


# either side of the lines between the fused kernels and the chain: rows, and
# blocks of 64 of them
@pytest.mark.parametrize("H,T,hd", [(1, 512, 96), (1, 513, 96), (12, 600, 96), (13, 600, 96), (1, 128, 128),
                                    (1, 129, 128), (76, 310, 128), (77, 310, 128)])
def test_both_sides_of_the_lines(dev, H, T, hd):
    P = Pico()
    xs = np.random.default_rng(T + H).standard_normal((3, T, H * hd)).astype(np.float32)
    with P.arena(1 << 30):
        q, k, v = (P.param([T, H * hd], x) for x in xs)
        y = P.attention_causal(q, k, v, 1, H)
        P.backward(y)
        out, grads = P.data(y), [P.grad(x) for x in (q, k, v)]
        for x in (q, k, v):
            P.free(x)
    q, k, v = (torch.from_numpy(x).to(dev) for x in xs)
    ro, _, rg = _reference(1, H, T, hd, q, k, v, torch.ones_like(q))
    _close(torch.from_numpy(out).to(dev).reshape(ro.shape), ro)
    for got, want in zip(grads, rg):
        err = (torch.from_numpy(got).to(dev).reshape(want.shape).double() - want).norm()
        # (the upstream of ones makes q's and k's exact gradients nearly cancel)
        assert float(err) <= TOL * float(rg[2].norm())


def test_refusals(dev):
    L = _lib.hip_lib()
    x = torch.zeros(64, 256, device=dev)
    lse = torch.zeros(64, device=dev)
    args = [_ptr(x)] * 4 + [_ptr(lse), None]
    for B, H, T, hd, ld in ((1, 1, 64, 64, 64), (1, 1, 64, 48, 48), (1, 1, 64, 96, 95), (1, 1, 64, 96, 98)):
        assert L.pk_flash_wide_fwd_f32(B, H, T, hd, ld, 1.0, *args) == -1
    assert L.pk_flash_wide_bwd_f32(1, 1, 64, 96, 96, 1.0, *([_ptr(x)] * 4), _ptr(lse), *([_ptr(x)] * 4),
                                   _ptr(x), 16, 0, None) == -1
    assert not L.pk_flash_wide_supported(64, 64) and L.pk_flash_wide_supported(1, 128)


# leading keys (more than a block of them) that no later query sees: scores of -inf, and
# scores next to which the others' would vanish.  The first 40 rows of the finite case
# see equal keys only, so their probabilities are equal too
@pytest.mark.parametrize("hd", [32, 96, 128])
@pytest.mark.parametrize("B,H,T", [(2, 3, 200), (16, 16, 130)])
@pytest.mark.parametrize("low", [float("-inf"), -1e30])
def test_leading_keys_far_below_the_others(dev, hd, B, H, T, low):
    g = torch.Generator(device=dev).manual_seed(T + hd)
    D, n = H * hd, 40
    q, k, v = (torch.randn(B * T, D, device=dev, generator=g) for _ in range(3))
    q = q.abs() + 0.01
    k.view(B, T, D)[:, :n] = low
    o, lse = _fwd(B, H, T, hd, D, q, k, v)
    x = [t.double().reshape(B, T, H, hd).transpose(1, 2).reshape(B * H, T, hd) for t in (q, k, v)]
    s = torch.bmm(x[0][:, n:].contiguous(), x[1][:, n:].transpose(1, 2).contiguous()) * hd ** -0.5
    s = s.masked_fill(~torch.ones(T - n, T - n, dtype=torch.bool, device=dev).tril(), float("-inf"))
    heads = o.reshape(B, T, H, hd).transpose(1, 2).reshape(B * H, T, hd)
    _close(heads[:, n:], torch.bmm(torch.softmax(s, -1), x[2][:, n:].contiguous()))
    _close(lse.reshape(B * H, T)[:, n:], torch.logsumexp(s, -1))
    if low > float("-inf"):
        count = torch.arange(1, n + 1, device=dev)[:, None]
        _close(heads[:, :n], x[2][:, :n].cumsum(1) / count)
    else:
        assert bool(torch.isnan(heads[:, :n]).all())
