"""fp8 appends with RoPE / PRoPE copies: raw frames and copies run together on the tile grids with a
workspace of the reported size, and after one another with a smaller one (which frames past 4096
tokens allow: the one-pass raw append's cells take less).  Codes and scales must not depend on which."""

import ctypes

import pytest
import torch

from solarwm_amd import _lib, kernels, rope

pytestmark = pytest.mark.gpu
F8 = torch.float8_e4m3fn


@pytest.mark.parametrize("B,H,gh,gw,n,prope,norm,dtype", [
    (1, 2, 70, 64, 1, False, False, torch.bfloat16),
    (2, 1, 70, 64, 2, True, True, torch.bfloat16),
    (1, 1, 75, 62, 1, True, False, torch.float32),   # 73 tiles, the last of 42 rows
    (1, 3, 80, 65, 1, False, True, torch.float32),   # 82 tiles: more than a wave's lanes
])
def test_joint_and_separate_passes_agree(gpu, B, H, gh, gw, n, prope, norm, dtype):
    print("joint append", B, H, gh, gw, n, prope, norm, dtype, flush=True)
    T = gh * gw
    g = torch.Generator(device=gpu).manual_seed(T)
    k, v = (torch.randn(B, n * T, H, 128, generator=g, device=gpu).to(dtype) for _ in range(2))
    hw = rope.spatial_table(rope.RopeConfig(grid_hw=(gh, gw)), gpu)
    xf = torch.randn(n, B, 4, 4, generator=g, device=gpu)
    w = torch.rand(H * 128, generator=g, device=gpu) + 0.5
    results = []
    for joint in (True, False):
        kp, vp, ks, vs = kernels.new_pools(n, B, H, T, F8, gpu)
        kr, vr = torch.zeros_like(kp), torch.zeros_like(vp)
        krs, vrs = torch.zeros_like(ks), torch.zeros_like(vs)
        kw = dict(vr_pool=vr, kv_xform=xf, vr_scale=vrs) if prope else {}
        launch = kernels.prepare_append(
            k, v, kp, vp, list(range(n)), frame_tokens=T, kscale=ks, vscale=vs, kr_pool=kr,
            rope_hw=hw, grid_hw=(gh, gw), kr_scale=krs,
            k_norm=(kernels.rms_rows(k, 1e-6), w) if norm else None, **kw)
        (desc,) = [x for x in launch.keep if isinstance(x, _lib.AppendDesc)]
        need = ctypes.c_int64(0)
        _lib.check("size", _lib.load().skv_append_workspace_size(ctypes.byref(desc), ctypes.byref(need)))
        units, tiles = 2 * n * B * H, -(-T // 64)
        assert need.value == 8 * units * tiles  # both sets of tile maxima
        size = need.value if joint else need.value - 4
        buf = torch.empty(size, dtype=torch.uint8, device=gpu)
        desc.workspace, desc.workspace_bytes = buf.data_ptr(), size
        launch()
        torch.cuda.synchronize()
        results.append([x.view(torch.uint8) for x in (kp, vp, kr, vr)] + [ks, vs, krs, vrs])
    for a, b in zip(*results):
        assert torch.equal(a, b)
    assert float(results[0][6].min()) > 0 and (not prope or float(results[0][7].min()) > 0)
