"""Frames in host memory reach the device through pinned slots of 1 MiB: the
device's copy has the host's bytes for row pitches with and without padding and
for images below, at and above a slot, and the caller's memory is free as soon
as the call returns.  A device frame's depth is too, and the Python loops hold
on to its colour until the next call."""
import ctypes

import numpy as np
import pytest

from slam_amd import synth
from slam_amd.frame_loop import BatchFrameLoop, FrameLoop, LoopParams
from slam_amd.odometry import FMT_RGBA32F, MEM_HOST, FrameView, RGBDOdometry, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,pad", [(64, 48, 0), (256, 256, 0), (257, 255, 0), (333, 251, 16), (640, 480, 48)])
def test_uploaded_maps_equal_the_device_path(w, h, pad):
    import torch
    rng = np.random.default_rng(w)
    maps = [rng.normal(size=(h, w, 4)).astype(np.float32) + 2.0 for _ in range(2)]
    pose = np.eye(4, dtype=np.float32)
    args = (w, h, w / 2.0, h / 2.0, 0.8 * w, 0.8 * w)
    dev, host = RGBDOdometry(*args), RGBDOdometry(*args)
    dev.initICPModel(*[torch.from_numpy(m).cuda() for m in maps], 20.0, pose)
    pitch = w * 16 + pad
    views, keep = [], []
    for m in maps:
        rows = np.full((h, pitch), 0xAB, np.uint8)
        rows[:, :w * 16] = m.view(np.uint8).reshape(h, w * 16)
        keep.append(rows)
        views.append(FrameView(rows.ctypes.data, pitch, w, h, FMT_RGBA32F, MEM_HOST))
    p = np.ascontiguousarray(pose.reshape(16))
    assert lib().odom_init_icp_model(host._h, ctypes.byref(views[0]), ctypes.byref(views[1]), 20.0,
                                     p.ctypes.data_as(ctypes.POINTER(ctypes.c_float))) == 0
    for rows in keep:
        rows[:] = 0                       # the call has taken its copy
    for name in ("vmap_g_prev", "nmap_g_prev"):
        for level in range(3):
            a, b = dev.read_buffer(name, level), host.read_buffer(name, level)
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (name, level)


def test_loop_over_host_frames_equals_device_frames():
    import torch
    cam = synth.CAM_320
    scene = synth.Scene(3)
    poses = synth.spline_trajectory(5, seed=3)
    frames = [scene.render(T, cam, noise_seed=k, model=False) for k, T in enumerate(poses)]
    args = (cam.width, cam.height, cam.cx, cam.cy, cam.fx, cam.fy)
    host, dev = (FrameLoop(*args, LoopParams(max_surfels=300_000)) for _ in range(2))
    for f in frames:
        rgb, depth = f.rgb.copy(), f.depth.copy()
        a = host.process(rgb, depth)
        rgb[:], depth[:] = 0, 0
        b = dev.process(torch.from_numpy(f.rgb).cuda(), torch.from_numpy(f.depth).cuda())
        assert np.array_equal(a, b)
    assert np.array_equal(host.model.model().view(np.uint32), dev.model.model().view(np.uint32))


@pytest.mark.parametrize("n", [1, 3])
def test_loop_leaves_device_frames_alone_after_the_call(n):
    """Depth tensors are overwritten as soon as the call returns, colour
    tensors are dropped and their size is allocated and filled again."""
    import torch
    cam = synth.CAM_640
    scene = synth.Scene(9)
    poses = synth.spline_trajectory(5, seed=9, max_step_m=0.01, max_step_deg=0.5)
    frames = [scene.render(T, cam, noise_seed=k, model=False) for k, T in enumerate(poses)]
    args = (cam.width, cam.height, cam.cx, cam.cy, cam.fx, cam.fy)
    p = LoopParams(max_surfels=1_500_000)
    make = (lambda: FrameLoop(*args, p)) if n == 1 else (lambda: BatchFrameLoop(n, *args, p))
    host, dev = make(), make()
    for f in frames:
        rgbs = [torch.from_numpy(f.rgb).cuda() for _ in range(n)]
        depths = [torch.from_numpy(f.depth).cuda() for _ in range(n)]
        torch.cuda.synchronize()
        if n == 1:
            a, b = host.process(f.rgb, f.depth), dev.process(rgbs[0], depths[0])
        else:
            a, b = host.process([f.rgb] * n, [f.depth] * n), dev.process(rgbs, depths)
        for d in depths:
            d.fill_(1000)
        del rgbs
        again = [torch.full(f.rgb.shape, 77, dtype=torch.uint8, device="cuda") for _ in range(2 * n)]
        assert np.array_equal(np.asarray(a), np.asarray(b))
        del again
    models = [(host.model, dev.model)] if n == 1 else list(zip(host.models, dev.models))
    for x, y in models:
        assert np.array_equal(x.model().view(np.uint32), y.model().view(np.uint32))


def test_host_frames_allocate_no_device_memory():
    """The loop's and the handles' memory is theirs from create on: the first
    host frames take none."""
    import torch
    w, h = 1920, 1080
    args = (w, h, w / 2.0, h / 2.0, 0.8 * w, 0.8 * w)
    rgb = np.full((h, w, 3), 90, np.uint8)
    depth = np.full((h, w), 1500, np.uint16)
    loop, odo = FrameLoop(*args, LoopParams(max_surfels=3_000_000, use_graph=False)), RGBDOdometry(*args)
    warm = FrameLoop(64, 48, 32.0, 24.0, 50.0, 50.0, LoopParams(max_surfels=10_000, use_graph=False))
    for _ in range(2):                       # the runtime's own pools
        warm.process(rgb[:48, :64].copy(), depth[:48, :64].copy())
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    odo.initFirstRGB(rgb)
    for _ in range(2):
        loop.process(rgb, depth)
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == free
