"""The pyramid and model map launches where their tiles end: sizes at, just below and just
above a tile (64x32 level-0 texels), odd halvings, the smallest handle, and
three- and four-byte colour with padded rows, bit for bit against the oracle.
Depth and intensity have holes, steps beyond the 3-sigma gate and the largest
16-bit values, so every kind of tap is met at every edge."""
import ctypes

import numpy as np
import pytest

from slam_amd import synth
from slam_amd.odometry import (FMT_RGB8, FMT_RGBA8, MEM_HOST, FrameView, RGBDOdometry, _check, lib)

pytestmark = pytest.mark.gpu

SIZES = [(16, 16), (63, 31), (64, 32), (65, 33), (66, 35), (128, 64), (131, 97), (190, 66)]


def inputs(w, h, ch):
    rng = np.random.default_rng(1000 * w + h + ch)
    depth = rng.integers(900, 960, (h, w)).astype(np.uint16)
    depth[rng.random((h, w)) < 0.1] = 0
    depth[rng.random((h, w)) < 0.1] += 400
    depth[rng.random((h, w)) < 0.02] = 65535
    depth[:, -1] = 65535                      # next to texels outside the image
    v4 = rng.uniform(0.3, 7.0, (h, w, 4)).astype(np.float32)
    v4[rng.random((h, w)) < 0.15, 2] = 0.0
    v4[rng.random((h, w)) < 0.02, 2] = np.nan
    v4[: h // 3, : w // 3, 2] = 0.0           # windows without a valid texel
    rgb = rng.integers(0, 256, (h, w, ch)).astype(np.uint8)
    rgb[rng.random((h, w)) < 0.2] = 0
    rgb[h // 2:, : w // 2] = 0
    return depth, v4, rgb


@pytest.mark.parametrize("ch,pad", [(3, 0), (3, 5), (4, 0), (4, 7)])
@pytest.mark.parametrize("w,h", SIZES)
def test_pyramids_at_tile_edges(orc, w, h, ch, pad):
    depth, v4, rgb = inputs(w, h, ch)
    cam = (w, h, (w - 1) / 2, (h - 1) / 2, 0.8 * w, 0.8 * w)
    gpu, ref = RGBDOdometry(*cam), orc.Odometry(*cam)
    n4 = np.random.default_rng(w).normal(size=v4.shape).astype(np.float32)
    T = synth.perturb(np.eye(4), np.random.default_rng(h), 0.5, 30.0).astype(np.float32)
    for o in (gpu, ref):
        o.initICPModel(v4, n4, 20.0, T)
        o.initICP(depth, 20.0)
    rows = np.full((h, w * ch + pad), 255, np.uint8)
    rows[:, :w * ch] = rgb.reshape(h, w * ch)
    view = FrameView(rows.ctypes.data, w * ch + pad, w, h, FMT_RGB8 if ch == 3 else FMT_RGBA8, MEM_HOST)
    for name in ("odom_init_rgb", "odom_init_rgb_model"):
        _check(name, getattr(lib(), name)(gpu.handle, ctypes.byref(view)))
    ref.initRGB(rgb)
    ref.initRGBModel(rgb)
    for l in range(3):
        for mine, theirs in (("next_image", "nextImage"), ("last_image", "lastImage"), ("next_depth", "nextDepth"),
                             ("last_depth", "lastDepth"), ("depth", "depth_tmp"), ("vmap_curr", "vmap_curr"),
                             ("nmap_curr", "nmap_curr"), ("vmap_g_prev", "vmap_g_prev"),
                             ("nmap_g_prev", "nmap_g_prev")):
            if mine == "depth" and l == 0:
                continue                      # the input
            a, b = gpu.read_buffer(mine, l), np.asarray(ref.buf(theirs, l)).reshape(gpu.read_buffer(mine, l).shape)
            if a.dtype == np.float32:
                assert np.array_equal(np.isnan(a), np.isnan(b)), (mine, l)
                a, b = np.nan_to_num(a), np.nan_to_num(b)
            assert np.array_equal(a, b), (mine, l, np.argwhere(a != b)[:4])


@pytest.mark.parametrize("w,h", [(704, 496), (705, 497), (1025, 343), (577, 607)])
def test_model_maps_of_both_forms(orc, w, h):
    """From 350 000 pixels on a workgroup forms all levels of a 64x16 tile,
    below it level 1 has workgroups of its own: sizes on both sides of the
    line, the tiles' remainders, with a transform and without."""
    _, v4, _ = inputs(w, h, 3)
    n4 = np.random.default_rng(w).normal(size=v4.shape).astype(np.float32)
    T = synth.perturb(np.eye(4), np.random.default_rng(h), 0.5, 30.0).astype(np.float32)
    cam = (w, h, (w - 1) / 2, (h - 1) / 2, 0.8 * w, 0.8 * w)
    gpu, ref = RGBDOdometry(*cam), orc.Odometry(*cam)
    for o in (gpu, ref):
        o.initICPModel(v4, n4, 20.0, T)
        o.initICPMaps(n4, v4, 20.0)
    for l in range(3):
        for name in ("vmap_curr", "nmap_curr", "vmap_g_prev", "nmap_g_prev"):
            a = gpu.read_buffer(name, l)
            b = np.asarray(ref.buf(name, l)).reshape(a.shape)
            assert np.array_equal(np.isnan(a), np.isnan(b)), (name, l)
            assert np.array_equal(np.nan_to_num(a), np.nan_to_num(b)), (name, l)


@pytest.mark.parametrize("w", [16, 65])
def test_last_texel_of_a_device_image(orc, w):
    """Three-byte colour on the device, whose last texel is read from the byte
    before it: level 0 against the conversion's own expression, every level
    against the oracle.  (That no read leaves the image is checked on the CPU,
    in test_image_reads.py.)"""
    import torch
    h = 32
    rgb = torch.randint(1, 256, (h, w, 3), dtype=torch.uint8, generator=torch.Generator().manual_seed(w))
    cam = (w, h, w / 2, h / 2, 0.8 * w, 0.8 * w)
    gpu, ref = RGBDOdometry(*cam), orc.Odometry(*cam)
    v4 = np.ones((h, w, 4), np.float32)
    for o, img in ((gpu, rgb.cuda()), (ref, rgb.numpy())):
        o.initICPModel(v4, v4, 20.0, np.eye(4, dtype=np.float32))
        o.initRGB(img)
    c = rgb.numpy().astype(np.float32)
    plain = (c[..., 0] * np.float32(0.114) + c[..., 1] * np.float32(0.299) + c[..., 2] * np.float32(0.587))
    assert np.array_equal(gpu.read_buffer("next_image", 0), plain.astype(np.uint8))
    for l in range(3):
        a = gpu.read_buffer("next_image", l)
        assert np.array_equal(a, np.asarray(ref.buf("nextImage", l)).reshape(a.shape)), l
