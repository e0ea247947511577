"""float32 chunks staged into bf16 pools (``skv_append_round``): bit for bit the pools a bf16 append of
the rounded chunk writes, padding rows included, and the dense float32 attention built on it."""

import ctypes

import pytest
import torch

from oracle import wan_cache_ref as ref
from solarwm_amd import _lib, attention, kernels

from .helpers import assert_attn_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,T,n", [(1, 1, 1, 1), (2, 3, 63, 2), (1, 2, 64, 3), (2, 1, 65, 1), (1, 5, 405, 4)])
def test_rounded_pools_bit_exact(gpu, B, H, T, n):
    print("append round", B, H, T, n, flush=True)
    g = torch.Generator(device=gpu).manual_seed(T)
    # a padded token stride; the rounding's edge values: ties, overflow to infinity, infinities, NaN
    big = torch.randn(2, B, n * T, H, 144, generator=g, device=gpu)
    edge = torch.tensor([1.00390625, 1.01171875, 3.4e38, -3.4e38, float("inf"), float("nan"), 1e-40, -0.0],
                        device=gpu)
    big[:, :, : n * T, :, 8:16] = edge
    k, v = big[0, ..., :128], big[1, ..., :128]
    kernels.staging_pools(n, B, H, T, torch.bfloat16, gpu, torch.float32)[0].fill_(float("nan"))
    kp, vp = kernels.stage_frames(k, v, n, T)
    kp, vp = kp.clone(), vp.clone()
    wk, wv, _, _ = kernels.new_pools(n, B, H, T, torch.bfloat16, gpu)
    kernels.append_frames(k.bfloat16(), v.bfloat16(), wk, wv, list(range(n)), frame_tokens=T)
    torch.cuda.synchronize()
    for got, want in ((kp, wk), (vp, wv)):
        nan = want.isnan()
        assert torch.equal(got.isnan(), nan)
        assert torch.equal(got.view(torch.int16)[~nan], want.view(torch.int16)[~nan])


def test_float32_and_bf16_calls_stage_apart(gpu):
    """float32 K/V rounded to bf16 go to a buffer of their own: staging them leaves bf16 frames staged
    on the same stream (by another thread, say) as they are."""
    x = torch.randn(1, 64, 2, 128, device=gpu)
    kp, vp = kernels.stage_frames(x.bfloat16(), x.bfloat16(), 1, 64)
    before = kp.clone(), vp.clone()
    kr, _ = kernels.stage_frames(x + 1, x + 1, 1, 64)
    assert kr.data_ptr() != kp.data_ptr()
    assert torch.equal(kp, before[0]) and torch.equal(vp, before[1])


def test_round_refuses_other_types(gpu):
    k32 = torch.zeros(1, 64, 1, 128, device=gpu)
    for src, pool in ((torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32),
                      (torch.float16, torch.bfloat16)):
        kp, vp, _, _ = kernels.new_pools(1, 1, 1, 64, pool, gpu)
        with pytest.raises(ValueError):
            kernels.prepare_append(k32.to(src), k32.to(src), kp, vp, [0], frame_tokens=64,
                                   entry="skv_append_round")()
    kp, vp, _, _ = kernels.new_pools(1, 1, 1, 64, torch.bfloat16, gpu)
    with pytest.raises(ValueError):  # the plain append still refuses the conversion
        kernels.append_frames(k32, k32, kp, vp, [0], frame_tokens=64)
    with pytest.raises(ValueError):
        kernels.prepare_append(k32, k32, kp, vp, [0], frame_tokens=64, entry="skv_append_round",
                               k_norm=(torch.ones(1, 64, device=gpu), torch.ones(128, device=gpu)))()
    assert _lib.load().skv_append_round(ctypes.cast(None, ctypes.POINTER(_lib.AppendDesc)), None) == _lib.SKV_E_ARG


@pytest.mark.parametrize("B,H,Lq,Lk", [(1, 12, 1170, 4000), (2, 3, 70, 61), (1, 2, 300, 1024)])
def test_float32_dense_attention(gpu, B, H, Lq, Lk):
    print("dense f32", B, H, Lq, Lk, flush=True)
    g = torch.Generator().manual_seed(Lk)
    q = torch.randn(B, Lq, H, 128, generator=g)
    k, v = torch.randn(B, Lk, H, 128, generator=g), torch.randn(B, Lk, H, 128, generator=g)
    got = attention(q.to(gpu), k.to(gpu), v.to(gpu))
    assert got.dtype == torch.float32
    assert_attn_close(got, ref.attention(q.bfloat16(), k.bfloat16(), v.bfloat16()))
