"""The workgroup shape of unsplit attention launches (``skv_attention_plan``, no GPU needed: 256 CUs):
4-wave groups for short windows over grids that leave CUs idle, and for windows of up to 4 tiles; on
the GPU, that the rows around 128-row groups come out as the oracle has them."""

import pytest
import torch

from oracle import wan_cache_ref as ref
from solarwm_amd import _lib, kernels

from .helpers import assert_attn_close
from .test_capi import _attn_desc, _plan


@pytest.mark.parametrize("B,H,Lq,T,nf,pool,want", [
    (1, 24, 1215, 512, 1, _lib.SKV_BF16, 4),    # 240 groups of 128 rows, 8 tiles
    (1, 24, 1280, 640, 10, _lib.SKV_BF16, 4),   # 240 groups, 100 tiles
    (1, 2, 16384, 6464, 1, _lib.SKV_BF16, 8),   # 256 groups, 101 tiles
    (1, 2, 16385, 512, 1, _lib.SKV_BF16, 8),    # 258 groups
    (1, 12, 4680, 512, 1, _lib.SKV_BF16, 8),    # 228 8-wave groups fill the chip
    (1, 12, 4680, 256, 1, _lib.SKV_BF16, 4),    # 4 tiles
    (1, 12, 4680, 257, 1, _lib.SKV_BF16, 8),    # 5 tiles
    (1, 2, 128, 64, 5, _lib.SKV_FP8_E4M3, 4),
    (1, 100, 256, 64, 70, _lib.SKV_BF16, 4),    # 200 groups over 229 MB of K and V
    (1, 110, 256, 64, 70, _lib.SKV_BF16, 8),    # 252 MB
    (1, 110, 256, 64, 70, _lib.SKV_FP8_E4M3, 4),
    (1, 30, 256, 64, 40, _lib.SKV_F32, 4),      # float32 pools: up to 40 tiles on under half the CUs
    (1, 30, 256, 64, 41, _lib.SKV_F32, 8),
    (1, 63, 256, 64, 41, _lib.SKV_F32, 8),
    (1, 64, 256, 64, 41, _lib.SKV_F32, 4),
    (1, 64, 1024, 64, 4, _lib.SKV_F32, 8),      # 512 groups: no short-window rule in one round
    (1, 40, 25600, 64, 2, _lib.SKV_F32, 4),     # many rounds, 2 tiles
    (1, 40, 6400, 64, 4, _lib.SKV_F32, 8),      # 3 or 4 tiles: 2000 groups
    (1, 256, 1536, 64, 4, _lib.SKV_F32, 8),     # 3072
    (1, 256, 1537, 64, 4, _lib.SKV_F32, 4),     # 3328
])
def test_waves_per_group(B, H, Lq, T, nf, pool, want):
    d, _keep = _attn_desc(B, H, Lq, T, nf, pool)
    plan = _plan(d)
    rows = 32 * want
    assert plan.waves_per_group == want and plan.split == 0
    assert plan.n_workgroups == plan.n_qtiles == -(-Lq // rows) * H * B


def test_waves_per_group_of_other_launches():
    """Chunk-causal float32 windows keep the longer line; fp8 frames decoded for PRoPE follow the
    float32 rule while all groups run at once."""
    d, _keep = _attn_desc(1, 4, 6016, 64, 94, _lib.SKV_F32, mask=_lib.SKV_MASK_CHUNK_CAUSAL)
    assert _plan(d).waves_per_group == 4
    for H, want in ((100, 4), (200, 8), (300, 4)):
        d, _keep = _attn_desc(1, H, 192, 64, 2, _lib.SKV_FP8_E4M3)
        fake = d.q
        d.rope_hw, d.grid_h, d.grid_w, d.n_qframes = fake, 8, 8, 3
        d.q_xform_t = d.q_xform_s = d.out_xform = fake
        assert _plan(d).waves_per_group == want, H
        d.q_xform_t = d.q_xform_s = d.out_xform = None
        d.rope_t = fake  # on the fp8 matrix cores: 4 tiles and fewer on any grid
        assert _plan(d).waves_per_group == 4


@pytest.mark.gpu
@pytest.mark.parametrize("H,Lq,T,nf", [(2, 1, 64, 1), (3, 127, 65, 2), (1, 129, 40, 3), (2, 257, 200, 4)])
def test_small_grids(gpu, H, Lq, T, nf):
    print("group shape", H, Lq, T, nf, flush=True)
    g = torch.Generator().manual_seed(Lq)
    q = torch.randn(1, Lq, H, 128, generator=g).bfloat16()
    k, v = (torch.randn(1, nf * T, H, 128, generator=g).bfloat16() for _ in range(2))
    kp, vp, _, _ = kernels.new_pools(nf, 1, H, T, torch.bfloat16, gpu)
    kernels.append_frames(k.to(gpu), v.to(gpu), kp, vp, list(range(nf)), frame_tokens=T)
    qd = q.to(gpu)
    assert kernels.attention_plan(qd, kp, vp, list(range(nf)), frame_tokens=T)["waves_per_group"] == 4
    out = kernels.attention_frames(qd, kp, vp, list(range(nf)), frame_tokens=T)
    torch.cuda.synchronize()
    assert_attn_close(out, ref.attention(q, k, v))
