"""RoPE on load at the edges of its launches: frames just under, at and over 64 tokens (below 64 the
temporal angles come straight from memory, from 64 on they are staged in LDS for at most five query
frames per q-tile), q-tiles that span five query frames, rows past the last q-tile, float32 queries
and the query RMSNorm, on the unsplit launch and on shares of the key split (whose segments start
inside frames and leave a remainder).  Against the oracle's float64 window RoPE; the bars are those
of tests/helpers.py, since the arithmetic is that of every bf16 attention instance."""

import pytest
import torch

from oracle import wan_cache_ref as ref
from solarwm_amd import kernels, rope

from .helpers import assert_attn_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gh,gw,n,nq,H,dtype,norm,split", [
    (4, 8, 5, 5, 2, torch.bfloat16, False, False),      # 32 tokens: 160 rows over 5 frames
    (7, 9, 70, 5, 15, torch.float32, True, True),       # 63 tokens, 2 q-tiles per head, 1-tile frames
    (8, 8, 7, 7, 2, torch.bfloat16, True, False),       # 64 tokens: a q-tile of 5 query frames
    (8, 8, 66, 6, 9, torch.bfloat16, False, True),      # 1-tile frames, ring reused every frame
    (5, 13, 44, 5, 7, torch.float32, False, True),      # 65 tokens: 2 tiles, the second 1 key
    (15, 27, 18, 3, 3, torch.bfloat16, True, True),     # 405 tokens, shares start inside frames
])
def test_rope_on_load_edges(gpu, gh, gw, n, nq, H, dtype, norm, split):
    print("rope edges", gh, gw, n, nq, H, dtype, norm, split, flush=True)
    T, eps = gh * gw, 1e-6
    g = torch.Generator().manual_seed(gh * 100 + n)
    q = torch.randn((1, nq * T, H, 128), generator=g).to(dtype)
    k = torch.randn((1, n * T, H, 128), generator=g).to(torch.bfloat16)
    v = torch.randn((1, n * T, H, 128), generator=g).to(torch.bfloat16)
    w = torch.rand(H * 128, generator=g) + 0.5
    kpos = list(range(n))
    qpos = kpos[-nq:]
    f = ref.wan_rope_freqs()
    qn = ref.norm_heads(q, w, eps) if norm else q
    want = ref.attention(ref.rope_frames(qn, (gh, gw), qpos, f), ref.rope_frames(k, (gh, gw), kpos, f), v)
    cfg = rope.RopeConfig(grid_hw=(gh, gw))
    hw, tt = rope.spatial_table(cfg, gpu), rope.temporal_table(qpos, kpos, cfg, gpu)
    kp, vp, _, _ = kernels.new_pools(n, 1, H, T, torch.bfloat16, gpu)
    krp = torch.zeros_like(kp)
    for j in range(0, n, 16):
        m = min(16, n - j)
        kernels.append_frames(k.to(gpu), v.to(gpu), kp, vp, list(range(j, j + m)), frame_tokens=T,
                              src_frame0=j, kr_pool=krp, rope_hw=hw, grid_hw=(gh, gw))
    qd = q.to(gpu)
    args = dict(frame_tokens=T, rope=(hw, (gh, gw), tt),
                q_norm=(kernels.rms_rows(qd, eps), w.to(gpu)) if norm else None)
    slots = list(range(n))
    assert (kernels.attention_plan(qd, krp, vp, slots, **args)["split"] == 1) == split
    for ws in (True, False):
        out = kernels.attention_frames(qd, krp, vp, slots, use_workspace=ws, **args)
        torch.cuda.synchronize()
        assert_attn_close(out, want)


@pytest.mark.parametrize("norm,split", [(False, False), (True, True)])
def test_rope_table_at_any_float(gpu, norm, split):
    """A temporal table that starts 4, 8 or 12 bytes past a 16-byte boundary (a contiguous slice of a
    larger tensor) gives what an aligned one gives: the instance that reads it from memory does the
    same arithmetic, up to contractions in the query's float32 turn (bf16 rounding of the turned query
    and of P: 2^-9 relative each)."""
    gh, gw, n, nq, H = 8, 9, 40, 4, 7 if split else 2
    T = gh * gw
    g = torch.Generator(device=gpu).manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
    q, w = rnd(1, nq * T, H, 128).bfloat16(), torch.rand(H * 128, generator=g, device=gpu) + 0.5
    k, v = rnd(1, n * T, H, 128).bfloat16(), rnd(1, n * T, H, 128).bfloat16()
    cfg = rope.RopeConfig(grid_hw=(gh, gw))
    hw, tt = rope.spatial_table(cfg, gpu), rope.temporal_table(range(n - nq, n), range(n), cfg, gpu)
    kp, vp, _, _ = kernels.new_pools(n, 1, H, T, torch.bfloat16, gpu)
    krp = torch.zeros_like(kp)
    kernels.append_frames(k, v, kp, vp, range(n), frame_tokens=T, kr_pool=krp, rope_hw=hw, grid_hw=(gh, gw))
    kw = dict(frame_tokens=T, q_norm=(kernels.rms_rows(q, 1e-6), w) if norm else None)
    assert (kernels.attention_plan(q, krp, vp, range(n), rope=(hw, (gh, gw), tt), **kw)["split"] == 1) == split
    want = kernels.attention_frames(q, krp, vp, range(n), rope=(hw, (gh, gw), tt), **kw).float()
    big = torch.empty(tt.numel() + 4, device=gpu)
    assert tt.data_ptr() % 16 == 0 and big.data_ptr() % 16 == 0
    for off in (1, 2, 3):
        moved = big[off : off + tt.numel()].view(tt.shape)
        moved.copy_(tt)
        got = kernels.attention_frames(q, krp, vp, range(n), rope=(hw, (gh, gw), moved), **kw).float()
        assert float((got - want).norm()) <= 2.0 ** -8 * float(want.norm()), off


@pytest.mark.parametrize("H,Lq,T,n,dtype", [
    (1, 257 * 256 - 100, 64, 8, torch.bfloat16),    # 1 tail q-tile, 8 units over every CU: empty shares
    (3, 86 * 256, 72, 8, torch.float32),            # 2 tail q-tiles of 9 packed tiles
    (4, 1024, 64, 80, torch.bfloat16),              # q-tiles in 16 shares: several batches of records
])
def test_merge_of_few_and_many_records(gpu, H, Lq, T, n, dtype):
    """The merge of split q-tiles where shares are empty, hold a single tile, or are many per
    q-tile: every row against the unsplit launch of the same inputs.  Both round P to bf16 against
    another running max and, for bf16 outputs, the result: four roundings of rms 0.735 * 2^-7 /
    sqrt(12) = 1.6e-3 relative, 3.1e-3 together.  A row is one draw over its keys and 128 channels, so
    the bar is three times that, 1e-2 of the row's norm; a key tile lost or counted twice moves a row
    by sqrt(1 / tiles), 0.11 at 80 tiles."""
    print("merge", H, Lq, T, n, dtype, flush=True)
    g = torch.Generator(device=gpu).manual_seed(H + n)
    rnd = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
    q = rnd(1, Lq, H, 128).to(dtype)
    k, v = rnd(1, n * T, H, 128).to(torch.bfloat16), rnd(1, n * T, H, 128).to(torch.bfloat16)
    kp, vp, _, _ = kernels.new_pools(n, 1, H, T, torch.bfloat16, gpu)
    for j in range(n):
        kernels.append_frames(k, v, kp, vp, [j], frame_tokens=T, src_frame0=j)
    slots = list(range(n))
    assert kernels.attention_plan(q, kp, vp, slots, frame_tokens=T)["split"] > 0
    out = kernels.attention_frames(q, kp, vp, slots, frame_tokens=T)
    plain = kernels.attention_frames(q, kp, vp, slots, frame_tokens=T, use_workspace=False)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    moved = (out.float() - plain.float()).norm(dim=-1) / plain.float().norm(dim=-1)
    assert float(moved.max()) <= 1e-2, float(moved.max())
