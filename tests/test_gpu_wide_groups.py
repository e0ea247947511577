"""Attention launches that only large grids make: 8-wave groups unsplit (a nearly full round of CUs),
and as shares of the key split and of a tail launch, over the instances that small grids run with 4
waves.  Against float64 attention of the pools' own contents (bars of tests/helpers.py): query rows
turned by their tables here, keys and values as the pools hold them (e4m3 frames decoded and rounded to
bf16, as these instances decode them), for heads from every part of the grid."""

import pytest
import torch

from solarwm_amd import kernels, rope

from .helpers import assert_attn_close

pytestmark = pytest.mark.gpu

BF, F16, F32, F8 = torch.bfloat16, torch.float16, torch.float32, torch.float8_e4m3fn


def _turn(x, cs, first):
    """Pairs first.. of x [..., 128] by cos, sin cs [..., pairs, 2]."""
    p = x[..., 2 * first : 2 * (first + cs.shape[-2])].unflatten(-1, (-1, 2))
    c, s = cs[..., 0].double(), cs[..., 1].double()
    out = torch.stack([p[..., 0] * c - p[..., 1] * s, p[..., 0] * s + p[..., 1] * c], -1).flatten(-2)
    return torch.cat([x[..., : 2 * first], out, x[..., 2 * (first + cs.shape[-2]) :]], -1)


def _want(q, k, v, T, kw):
    """float64 attention of one head: q [L, 128], k [n, T, 128], v [n, T, 128]."""
    L, n = q.shape[0], k.shape[0]
    tab, mode = kw.get("rope") or kw.get("prope"), "prope" if "prope" in kw else "rope" if "rope" in kw else ""
    if mode:
        hw, (gh, gw) = tab[0].view(gh_gw(tab), 21, 2), tab[1]
        t = torch.arange(L, device=q.device) % T
        f = torch.arange(L, device=q.device) // T
        q = _turn(q, torch.cat([hw[t // gw], hw[gh + t % gw]], 1), 22)
    scores = []
    for j in range(n):
        qj = q
        if mode == "rope":
            qj = _turn(q, tab[2][f, j], 0)
        elif mode == "prope":
            w, ps = tab[2][0, j][f].double(), tab[3][0][f].double()  # [L, 11, 4, 4], [L, 4, 4]
            x = q.unflatten(-1, (32, 4))
            qj = torch.cat([(w @ x[:, :11, :, None])[..., 0], (ps[:, None] @ x[:, 11:, :, None])[..., 0]], 1).flatten(1)
        scores.append(qj @ k[j].T)
    out = torch.softmax(torch.cat(scores, 1) / 128 ** 0.5, -1) @ v.flatten(0, 1)
    if mode == "prope":
        out = (tab[4][0][f].double()[:, None] @ out.unflatten(-1, (32, 4))[..., None])[..., 0].flatten(1)
    return out


def gh_gw(tab):
    return tab[1][0] + tab[1][1]


@pytest.mark.parametrize("mode,pool,qt,grid,n,nq,H,norm,waves,split", [
    ("prope", BF, BF, (8, 8), 6, 4, 240, True, 8, 0),
    ("prope", BF, F32, (8, 9), 5, 3, 240, False, 8, 0),   # 2 tiles a frame, 216 rows
    ("prope", F8, BF, (8, 8), 6, 4, 240, False, 8, 0),
    ("rope", BF, BF, (7, 9), 6, 4, 240, False, 8, 0),     # frames under 64 tokens
    ("rope", BF, F32, (7, 9), 6, 4, 240, True, 8, 0),
    ("rope", F8, BF, (7, 9), 6, 4, 240, False, 8, 0),
    ("rope", BF, F32, (8, 8), 6, 4, 240, True, 8, 0),
    ("", F32, BF, (8, 8), 6, 4, 240, False, 8, 0),
    ("", F32, F32, (8, 8), 6, 4, 240, True, 8, 0),
    ("prope", BF, F32, (8, 8), 30, 4, 95, True, 8, 1),
    ("prope", F8, BF, (8, 9), 20, 3, 95, True, 8, 1),
    ("rope", BF, BF, (7, 9), 30, 4, 95, True, 8, 1),
    ("rope", F8, BF, (7, 9), 30, 4, 95, True, 8, 1),
    ("", F32, BF, (8, 8), 30, 4, 95, False, 8, 1),
    ("", F16, F32, (8, 8), 30, 4, 95, False, 8, 1),
    ("", F16, F32, (8, 9), 30, 3, 95, False, 8, 1),       # packed tiles
    ("prope", BF, BF, (8, 8), 8, 4, 316, False, 8, 2),    # one round and a split tail of 60 q-tiles
    ("prope", F8, BF, (8, 8), 8, 4, 316, True, 8, 2),
    ("rope", BF, F32, (7, 9), 8, 4, 316, False, 8, 2),
    ("prope", BF, F32, (8, 8), 3, 2, 5, True, 4, 0),
])
def test_wide_grids(gpu, mode, pool, qt, grid, n, nq, H, norm, waves, split):
    print("wide grid", mode, pool, qt, grid, n, nq, H, norm, flush=True)
    T = grid[0] * grid[1]
    g = torch.Generator(device=gpu).manual_seed(H + n)
    rnd = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
    k, v = (rnd(1, n * T, H, 128).to(BF if pool == F8 else pool) for _ in range(2))
    kp, vp, ks, vs = kernels.new_pools(n, 1, H, T, pool, gpu)
    kw = dict(frame_tokens=T) | (dict(kscale=ks, vscale=vs) if pool == F8 else {})
    kernels.append_frames(k, v, kp, vp, range(n), **kw)
    if mode:
        cfg, eye = rope.RopeConfig(grid_hw=grid), torch.eye(4, device=gpu)
        hw = rope.spatial_table(cfg, gpu)
        kw[mode] = ((hw, grid, rope.temporal_table(range(n - nq, n), range(n), cfg, gpu)) if mode == "rope" else
                    (hw, grid, *(eye + 0.1 * rnd(*s, 4, 4) for s in ((1, n, nq, 11), (1, nq), (1, nq)))))
    q, w = rnd(1, nq * T, H, 128).to(qt), torch.rand(H * 128, generator=g, device=gpu) + 0.5
    inv = kernels.rms_rows(q, 1e-6) if norm else None
    args = dict(kw, q_norm=(inv, w) if norm else None)
    plan = kernels.attention_plan(q, kp, vp, range(n), **args)
    assert (plan["waves_per_group"], plan["split"]) == (waves, split), plan
    got = kernels.attention_frames(q, kp, vp, range(n), **args)
    for h in sorted({0, H // 7, H // 3, H // 2, H - 1 - H // 5, H - 2, H - 1}):
        kh, vh = kp[:, 0, h, :T], vp[:, 0, h, :, :T].transpose(1, 2)
        if pool == F8:
            kh, vh = (x.float() * sc[:, 0, h, None, None] for x, sc in ((kh, ks), (vh, vs)))
        half = torch.float16 if pool == F16 else BF  # what the matrix cores multiply
        x = q[0, :, h].float()
        x = x * inv[0, :, None] * w[h * 128 : h * 128 + 128] if norm else x.to(half)
        want = _want(x.double(), kh.to(half).double(), vh.to(half).double(), T, kw)
        assert_attn_close(got[0, :, h], want.cpu())
