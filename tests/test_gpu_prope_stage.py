"""The one-launch camera staging (skv_prope_stage) against the tensor operations of the same tables.

Both compute in float64 and round to float32 once, so they differ by one float32 rounding where the
order of a float64 sum falls on the other side of it, plus float64 noise where terms cancel."""

import ctypes

import pytest
import torch
from torch._subclasses import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx

from solarwm_amd import PropeConfig, RopeConfig, _lib, make_kv_cache_allocator, prope, stage_camera_cache

from .cameras import trajectory

T = 64


def _caches(dev, B, cap, sink, nb, transform, echo):
    return make_kv_cache_allocator(
        num_layers=1, num_heads=1, head_dim=128, frame_sequence_length=T, local_attn_size=cap,
        sink_size=sink, num_frame_per_block=nb, rope=RopeConfig(grid_hw=(8, 8), use_echorope=echo),
        prope=PropeConfig(camera_translation_transform=transform))(B, dtype=torch.bfloat16, device=dev)


def _close(got, want):
    got, want = got.double(), want.double()
    bound = want.abs() * 2.0**-23 + (2.0**-44 * want.abs().max() if want.numel() else 0.0)
    assert bool(((got - want).abs() <= bound).all()), float((got - want).abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("B,sink,cap,nb,schedule,transform,echo", [
    (2, 1, 6, 2, [0, 2, 4, 6, 8], "linear", True),
    (1, 0, 5, 1, [0, 1, 2, 3, 4, 5], "logd4", True),
    (2, 1, 5, 2, [0, 2, 2, 4, 6], "logd4", False),  # a recompute pass at frame 2
    (3, 2, 6, 2, [0, 2, 0, 4, 6], "linear", True),  # a recached sink keeps its cameras
    (1, 0, 60, 25, [0, 25, 50], "linear", False),  # over 256 (frame, group) pairs a block
])
def test_stage_kernel_matches_tensor_operations(gpu, monkeypatch, B, sink, cap, nb, schedule,
                                                transform, echo):
    vm, ks = (x.to(gpu) for x in trajectory(B, max(schedule) + nb, seed=7, t_scale=0.8))
    new, old = (_caches(gpu, B, cap, sink, nb, transform, echo) for _ in range(2))
    seen = []
    kernel = prope._stage_kernel
    monkeypatch.setattr(prope, "_stage_kernel", lambda *a: (seen.append(1), kernel(*a))[1])
    rule = prope._kernel_stages
    for i, f in enumerate(schedule):
        recache = i > 0 and f == 0
        args = dict(per_frame=True, sink_recache_after_switch=recache)
        monkeypatch.setattr(prope, "_kernel_stages", rule)
        a = stage_camera_cache(new, vm, ks, f * T, nb * T, **args)
        monkeypatch.setattr(prope, "_kernel_stages", lambda *a: False)
        b = stage_camera_cache(old, vm, ks, f * T, nb * T, **args)
        assert len(seen) == i + 1
        assert (a.staging, a.window) == (b.staging, b.window)
        for name in ("kv_xform", "q_xform_t", "q_xform_s", "out_xform"):
            x, y = getattr(a, name), getattr(b, name)
            assert x.shape == y.shape and x.is_contiguous() and x.dtype == y.dtype
            _close(x, y)
        assert torch.equal(new[0].camera.viewmats, old[0].camera.viewmats)
        assert torch.equal(new[0].camera.ks, old[0].camera.ks)
        _close(new[0].camera.p_inv, old[0].camera.p_inv)
        for c in (new[0], old[0]):
            plan, temp, staging, window = c.plan(f * T, nb * T, recache)
            c.commit(c.stage(plan, temp), plan.current_end, plan.local_end_index)


@pytest.mark.gpu
def test_stage_kernel_takes_strided_cameras(gpu):
    """Per-token cameras (frame stride T matrices), transposed matrices, expanded streams."""
    vm, ks = (x.to(gpu) for x in trajectory(1, 3, seed=9))
    want = stage_camera_cache(_caches(gpu, 2, 5, 0, 3, "linear", True), vm.repeat(2, 1, 1, 1),
                              ks.repeat(2, 1, 1, 1), 0, 3 * T, per_frame=True)
    tr = vm.transpose(-1, -2).contiguous().transpose(-1, -2)
    forms = [(vm.expand(2, -1, -1, -1), ks.expand(2, -1, -1, -1), True),
             (tr.expand(2, -1, -1, -1), ks.expand(2, -1, -1, -1), True),
             (vm.repeat_interleave(T, 1).repeat(2, 1, 1, 1), ks.repeat_interleave(T, 1).repeat(2, 1, 1, 1),
              False)]
    for v, k, per_frame in forms:
        got = stage_camera_cache(_caches(gpu, 2, 5, 0, 3, "linear", True), v, k, 0, 3 * T,
                                 per_frame=per_frame)
        for name in ("kv_xform", "q_xform_t", "q_xform_s", "out_xform"):
            assert torch.equal(getattr(got, name), getattr(want, name))


@pytest.mark.gpu
def test_staging_without_new_frames(gpu):
    """A call without new frames over a committed history gives empty query tables, as on the CPU."""
    vm, ks = trajectory(2, 2, seed=5)
    shapes = []
    for dev in (gpu, torch.device("cpu")):
        caches = _caches(dev, 2, 6, 1, 2, "linear", True)
        stage_camera_cache(caches, vm.to(dev), ks.to(dev), 0, 2 * T, per_frame=True)
        c = caches[0]
        plan, temp, _, _ = c.plan(0, 2 * T, False)
        c.commit(c.stage(plan, temp), plan.current_end, plan.local_end_index)
        got = stage_camera_cache(caches, vm.to(dev), ks.to(dev), 2 * T, 0, per_frame=True)
        shapes.append([tuple(getattr(got, n).shape) for n in ("kv_xform", "q_xform_t", "q_xform_s", "out_xform")])
    assert shapes[0] == shapes[1] and shapes[0][1] == (2, 2, 0, 11, 4, 4)


@pytest.mark.gpu
def test_followed_cameras_keep_what_follows_them(gpu):
    """Forward-mode tangents reach the four tables, and the gradients of cameras staged earlier reach
    the tables of later forwards through the store."""
    fwd = torch.autograd.forward_ad
    vm, ks = (x.to(gpu) for x in trajectory(1, 4, seed=3))
    tables = ("kv_xform", "q_xform_t", "q_xform_s", "out_xform")
    want = stage_camera_cache(_caches(gpu, 1, 5, 0, 2, "logd4", True), vm, ks, 0, 2 * T, per_frame=True)
    with fwd.dual_level():
        dual = fwd.make_dual(vm, torch.randn_like(vm))
        got = stage_camera_cache(_caches(gpu, 1, 5, 0, 2, "logd4", True), dual, ks, 0, 2 * T, per_frame=True)
        for name in tables:
            x = fwd.unpack_dual(getattr(got, name))
            assert x.tangent is not None and float(x.tangent.abs().max()) > 0, name
            _close(x.primal, getattr(want, name))
    caches = _caches(gpu, 1, 5, 0, 2, "linear", True)
    first = vm[:, :2].clone().requires_grad_()
    stage_camera_cache(caches, first, ks[:, :2], 0, 2 * T, per_frame=True)
    c = caches[0]
    plan, temp, _, _ = c.plan(0, 2 * T, False)
    c.commit(c.stage(plan, temp), plan.current_end, plan.local_end_index)
    later = stage_camera_cache(caches, vm, ks, 2 * T, 2 * T, per_frame=True)
    (grad,) = torch.autograd.grad(later.q_xform_t.sum(), first)
    assert float(grad.abs().max()) > 0


def test_stage_rule_and_refusals():
    cam = prope.CameraCache(8, 2, "cpu", PropeConfig())
    v, k = torch.zeros(2, 3, 4, 4), torch.zeros(2, 3, 3, 3)
    assert not prope._kernel_stages(cam, v, k, [0], [-1], 0, [0], [0, 1, 2])  # CPU cameras
    cam.device = torch.device("cuda", 0)  # the rule reads sizes and marks only

    def rule(v=v, k=k, staging=(4, 5, 6), keep=(-1, -1, 2), off=0, window=(0, 4), qpos=(5, 6, 7)):
        return prope._kernel_stages(cam, v, k, staging, keep, off, window, qpos)

    assert rule() and rule(qpos=(5, 5, 5))
    assert not rule(v=v[:1]) and not rule(k=torch.zeros(2, 3, 4, 4)) and not rule(off=1)
    assert not rule(keep=(-1, -1, 4)) and not rule(staging=(4, 5, 5)) and not rule(qpos=(5, 6, 8))
    assert not rule(v=v.to("meta")) and not rule(k=k.to("meta"))  # on another device than the store
    assert not rule(v=v[:, :0], k=k[:, :0], staging=(), keep=(), qpos=())  # no new frames
    wide = prope.CameraCache(1, 65536, "cpu", PropeConfig())
    wide.device = cam.device
    assert not prope._kernel_stages(wide, v[:1, :1].expand(65536, 1, 4, 4), k[:1, :1].expand(65536, 1, 3, 3),
                                    [0], [-1], 0, [0], [0])
    assert not rule(window=()) and not rule(window=range(257))
    assert not rule(v=v.clone().requires_grad_())


    # cameras, or a store, that something follows: the launch would lose it
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(v, torch.ones_like(v))
        assert not rule(v=dual) and not rule(k=torch.autograd.forward_ad.make_dual(k, torch.ones_like(k)))
    seen = []
    torch.func.vmap(lambda x: (seen.append(rule(v=x)), x)[1])(v[None])
    torch.func.jvp(lambda x: (seen.append(rule(k=x)), x)[1], (k,), (k,))
    make_fx(lambda x: (seen.append(rule(v=x)), x + 1)[1])(v)
    with FakeTensorMode() as fake:
        seen.append(rule())
        seen.append(rule(v=fake.from_tensor(v)))
    assert seen == [False] * 5 and rule()
    assert not rule(v=torch._neg_view(v))
    for name in ("viewmats", "ks", "p_inv"):
        t = getattr(cam, name)
        setattr(cam, name, t.clone().requires_grad_())
        assert not rule(), name
        setattr(cam, name, t)
    assert rule()

    lib = _lib.load()
    buf = (ctypes.c_float * 64)()
    p = ctypes.addressof(buf)

    def call(**over):
        a = dict(n_slots=4, batch=1, n_qframes=2, n_keys=1, n_staged=1, first=0, q_step=1)
        win, st, kp = over.pop("window", [0]), over.pop("staged", [1]), over.pop("keep", [-1])
        a.update(over)
        d = _lib.PropeStageDesc(
            view=p, view_t=p, ks=p, store_view=p, store_k=p, store_inv=p, kv_xform=p, q_xform_t=p,
            q_xform_s=p, out_xform=p, inv_freq=(ctypes.c_double * 22)(),
            window=_lib.int32_array(win), k_pos=_lib.int32_array([0] * len(win)),
            staged=_lib.int32_array(st), keep=_lib.int32_array(kp), **a)
        return lib.skv_prope_stage(ctypes.byref(d), None)

    for over in (dict(n_keys=0), dict(n_keys=257), dict(n_staged=65), dict(first=2), dict(batch=0),
                 dict(batch=65536), dict(window=[4]), dict(window=[-1]), dict(staged=[4]),
                 dict(keep=[4]), dict(keep=[1]), dict(n_staged=2, staged=[1, 1], keep=[-1, -1])):
        assert call(**over) == _lib.SKV_E_ARG, over
    assert lib.skv_prope_stage(None, None) == _lib.SKV_E_ARG


def test_stage_launch_runs_on_the_cameras_device(monkeypatch):
    """The launch is made with the store's device current, whatever device the caller has current."""
    current, launched = [], []

    class Device:
        def __init__(self, dev):
            self.dev = dev

        def __enter__(self):
            current.append(self.dev)

        def __exit__(self, *a):
            current.pop()

    class Lib:
        @staticmethod
        def skv_prope_stage(desc, stream):
            launched.append((list(current), stream))
            return _lib.SKV_OK

    monkeypatch.setattr(torch.cuda, "device", Device)
    monkeypatch.setattr(prope.kernels, "_stream", lambda dev: ("stream of", dev))
    monkeypatch.setattr(prope._lib, "load", lambda: Lib)
    cam = prope.CameraCache(8, 2, "cpu", PropeConfig())
    v, k = torch.zeros(2, 3, 4, 4), torch.zeros(2, 3, 3, 3)
    prope._stage_kernel(cam, 1e4, v, v, k, [4], [-1], 0, [0, 4], [1, 2, 3], [0, 1])
    assert launched == [([cam.p_inv.device], ("stream of", cam.p_inv.device))]


def test_stage_descriptor_layout(tmp_path):
    from .test_capi import test_descriptor_layout_matches_header as layout

    layout(tmp_path, "skv_prope_stage_desc", "PropeStageDesc")
