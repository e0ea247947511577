"""The balanced key split with as many shares as divide every q-tile evenly (fewer than the CUs, whose
grid the plan still reports) against float64 attention and the unsplit launch: 2, 3 and many shares a
q-tile, counts on both sides of the rule's line, bf16 / fp8 pools, float32 queries, a ragged last q-tile
and the shares of a tail launch.  Bars: tests/helpers.py."""

import ctypes

import pytest
import torch

from solarwm_amd import _lib, kernels, rope

from .helpers import assert_attn_close

pytestmark = pytest.mark.gpu

BF, F8 = torch.bfloat16, torch.float8_e4m3fn


@pytest.mark.parametrize("H,Lq,T,n,pool,split", [
    (120, 250, 64, 30, BF, 1),   # 2 shares a q-tile, 240 of 256
    (84, 256, 72, 27, BF, 1),    # 3, 252: packed tiles over frame edges
    (3, 700, 200, 40, BF, 1),    # 28, 252; last q-tile 188 of 256 rows
    (100, 250, 64, 30, BF, 1),   # 200 shares, 3.3 extra tiles: even
    (100, 129, 1024, 3, BF, 1),  # 200 shares, 5.3 extra tiles
    (96, 200, 2048, 3, BF, 1),   # 192 shares would take 12 extra tiles: one a CU
    (84, 250, 100, 8, F8, 1),
    (96, 200, 2048, 3, F8, 1),   # 12 extra tiles: even for fp8
    (3, 700, 200, 40, F8, 1),
    (207, 1024, 200, 20, BF, 2),  # three full rounds, then 60 q-tiles in 4 shares each
])
@pytest.mark.parametrize("qt", [BF, torch.float32])
def test_even_shares(gpu, H, Lq, T, n, pool, split, qt):
    print("even shares", H, Lq, T, n, pool, qt, flush=True)
    g = torch.Generator(device=gpu).manual_seed(H * Lq + T)
    qd = torch.randn(1, Lq, H, 128, generator=g, device=gpu).to(qt)
    kd, vd = (torch.randn(1, n * T, H, 128, generator=g, device=gpu).to(BF) for _ in range(2))
    kp, vp, ks, vs = kernels.new_pools(n, 1, H, T, pool, gpu)
    kw = dict(kscale=ks, vscale=vs) if pool == F8 else {}
    for f in range(n):
        kernels.append_frames(kd, vd, kp, vp, [f], frame_tokens=T, src_frame0=f, **kw)
    plan = kernels.attention_plan(qd, kp, vp, range(n), frame_tokens=T, **kw)
    assert plan["split"] == split, plan
    if split == 1:
        assert plan["n_workgroups"] == kernels.cu_count(gpu), plan
    out = kernels.attention_frames(qd, kp, vp, range(n), frame_tokens=T, **kw)
    plain = kernels.attention_frames(qd, kp, vp, range(n), frame_tokens=T, use_workspace=False, **kw)
    # A probability is rounded once, in each launch against another running max.  Roundings to m
    # mantissa bits err by 2^-m / sqrt(12) / x, x in [1, 2) log-uniform: rms 0.735 * 2^-m / sqrt(12),
    # which is the output's relative rms error too (random signs in V); two independent ones differ by
    # sqrt(2) of it: e4m3 (m = 3) 3.8e-2, bf16 (m = 7) 2.3e-3, the latter plus the output's rounding.
    diff = (out.float() - plain.float()).norm() / plain.float().norm()
    assert diff <= (3.8e-2 if pool == F8 else 4e-3), diff
    if pool == BF:
        q64, k64, v64 = (x[0].transpose(0, 1).double() for x in (qd.to(BF), kd, vd))
        for h in range(0, H, 7):  # every 7th head, one at a time: q-tiles of every share pattern
            want = torch.softmax(q64[h] @ k64[h].T / 128 ** 0.5, -1) @ v64[h]
            assert_attn_close(out[0, :, h], want.cpu())


def _instance(gpu, mode, pool, H, T, n, nq):
    """Random pools, query and tables of one attention instance; (query, K, V, kwargs)."""
    g = torch.Generator(device=gpu).manual_seed(H + n)
    rnd = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
    tp = kernels.padded_tokens(T)
    k, v = rnd(n, 1, H, tp, 128).to(pool), rnd(n, 1, H, 128, tp).to(pool)
    kw = dict(frame_tokens=T)
    if pool == F8:
        kw |= dict(kscale=torch.full((n, 1, H), 0.5, device=gpu), vscale=torch.full((n, 1, H), 0.5, device=gpu))
    if mode:
        gh = next(x for x in range(int(T ** 0.5), 0, -1) if T % x == 0)
        grid, eye = (gh, T // gh), torch.eye(4, device=gpu)
        hw = rope.spatial_table(rope.RopeConfig(grid_hw=grid), gpu)
        if mode == "rope":
            kw["rope"] = (hw, grid, rope.temporal_table(range(n - nq, n), range(n), rope.RopeConfig(grid_hw=grid), gpu))
        else:
            kw["prope"] = (hw, grid, *(eye + 0.1 * rnd(*s, 4, 4) for s in ((1, n, nq, 11), (1, nq), (1, nq))))
    return rnd(1, nq * T, H, 128).to(BF), k, v, kw


@pytest.mark.parametrize("mode,pool,T,nq,even,uneven", [
    ("", BF, 48, 5, 53, 60),              # 95 q-tiles: 190 even shares cost nt * 0.129 extra tiles
    ("", BF, 64, 4, 69, 71),
    ("", torch.float32, 128, 2, 31, 32),
    ("rope", BF, 64, 4, 54, 55),
    ("rope", BF, 128, 2, 34, 36),
    ("rope", BF, 48, 5, 22, 39),
    ("rope", F8, 64, 4, 46, 47),
    ("rope", F8, 128, 2, 23, 24),
    ("rope", F8, 192, 1, 23, 24),
    ("rope", F8, 448, 1, 19, 20),         # 96 q-tiles: nt * 0.125
    ("prope", BF, 64, 4, 46, 47),
    ("prope", BF, 128, 2, 34, 36),
    ("prope", F8, 128, 2, 27, 28),
    ("prope", F8, 448, 1, 8, 9),
    ("", F8, 64, 4, 108, 110),
    ("", F8, 128, 2, 64, 70),
])
def test_share_count_follows_the_instance(gpu, mode, pool, T, nq, even, uneven):
    """Workgroups that write records (the workspace starts as NaN), at frame counts on both sides of
    the instance's line, and the result against the unsplit launch (bounds of test_even_shares)."""
    H = 95 if T < 256 else 48  # 448-token queries take two q-tiles a head: 96
    n_q = H * -(-nq * T // 256)
    for n, want in ((even, 256 // n_q * n_q), (uneven, 256)):
        print("share count", mode, pool, T, n, flush=True)
        q, k, v, kw = _instance(gpu, mode, pool, H, T, n, nq)
        plain = kernels.attention_frames(q, k, v, range(n), use_workspace=False, **kw)
        d, out, keep = kernels.attention_desc(q, k, v, range(n), **kw)
        plan = _lib.LaunchPlan()
        lib = _lib.load()
        _lib.check("plan", lib.skv_attention_plan(ctypes.byref(d), ctypes.byref(plan)))
        n_cu = kernels.cu_count(gpu)
        ws = torch.full((plan.workspace_bytes // 4,), float("nan"), device=gpu)
        d.workspace, d.workspace_bytes = ws.data_ptr(), plan.workspace_bytes
        _lib.check("attention", lib.skv_attention_ex(ctypes.byref(d), torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        ml = ws[2 * n_cu * 256 * 128 :].view(n_cu, 2, 256, 2)
        wrote = (~ml[..., 0].isnan()).flatten(1).any(1)
        assert int(wrote.sum()) == want, (n, int(wrote.sum()))
        diff = (out.float() - plain.float()).norm() / plain.float().norm()
        assert diff <= (3.8e-2 if pool == F8 and mode != "prope" else 4e-3), diff
