"""Derivatives and source masks, one or four pixels of a row a thread, and the SO3
sums, four pixels at a time past the first three: widths of every remainder of
4 on every level, small images, and levels 2 of 3 to 10 pixels a thread,
against the oracle; and the pairs of a batch (one launch for all) against
single calls."""
import numpy as np
import pytest

from slam_amd import synth
from slam_amd.odometry import Batch, RGBDOdometry

from helpers import CUTOFF, make_pair, pose_of

pytestmark = pytest.mark.gpu


def camera(w, h):
    return synth.Camera(w, h, 0.82 * w, 0.82 * w, w / 2.0, h / 2.0)


def fed(odo, T0, f0, f1, filt):
    odo.initFirstRGB(f0.rgb)
    odo.initICPModel(f0.vert4, f0.norm4, CUTOFF, T0.astype(np.float32))
    odo.initRGBModel(f0.rgba)
    odo.initICP(filt, CUTOFF)
    odo.initRGB(f1.rgb)
    return odo


@pytest.mark.parametrize("w,h", [(36, 30), (37, 31), (42, 33), (47, 40), (64, 48), (203, 77)])
def test_masks_and_derivatives_equal_the_oracle(orc, w, h):
    cam = camera(w, h)
    args = (w, h, cam.cx, cam.cy, cam.fx, cam.fy)
    T0, T1, f0, f1 = make_pair(cam, 21)
    filt = orc.bilateral(f1.depth, 5.0)
    odos = [fed(RGBDOdometry(*args), T0, f0, f1, filt) for _ in range(3)]
    ref = fed(orc.Odometry(*args), T0, f0, f1, filt)
    odos[0].getIncrementalTransformation(T0[:3, 3], T0[:3, :3], False, 10.0, True, False, False)
    for o in odos[1:]:
        o.set_pose(T0[:3, 3], T0[:3, :3])
    Batch(odos[1:]).track(False, 10.0, True, False, False)
    ref.getIncrementalTransformation(T0[:3, 3], T0[:3, :3], False, 10.0, True, False, False)
    for level in range(3):
        a = [o.read_buffer("dxy", level) for o in odos]
        m = [o.read_buffer("zsrc", level).view(np.uint32) for o in odos]
        assert np.array_equal(a[0], a[1]) and np.array_equal(a[0], a[2]), level
        assert np.array_equal(m[0], m[1]) and np.array_equal(m[0], m[2]), level
        img = odos[0].read_buffer("next_image", level).astype(np.int32)
        check_level(img, odos[0].read_buffer("next_depth", level), a[0], odos[0].read_buffer("zsrc", level), level)


def check_level(img, depth, dxy, zsrc, level):
    """The reference's loops, pixel by pixel."""
    gsx = np.float32([0.52201, 0, -0.52201, 0.79451, 0, -0.79451, 0.52201, 0, -0.52201])
    gsy = np.float32([0.52201, 0.79451, 0.52201, 0, 0, 0, -0.52201, -0.79451, -0.52201])
    h, w = img.shape
    scale = np.float32((5.0, 3.0, 1.0)[level] ** 2 * 64.0)
    for y in range(h):
        for x in range(w):
            dx, dy, k = np.float32(0), np.float32(0), 8
            for j in range(max(y - 1, 0), min(y + 1, h - 1) + 1):
                for i in range(max(x - 1, 0), min(x + 1, w - 1) + 1):
                    dx, dy, k = dx + np.float32(img[j, i]) * gsx[k], dy + np.float32(img[j, i]) * gsy[k], k - 1
            assert tuple(dxy[y, x]) == (int(dx), int(dy)), (x, y)
            ok = x < w - 5 and y < h - 1 and np.all(img[max(y - 2, 0):y + 2, max(x - 2, 0):x + 2] > 0) and \
                np.float32(int(dx) ** 2 + int(dy) ** 2) >= scale and not np.isnan(depth[y, x])
            assert zsrc[y, x] == depth[y, x] if ok else np.isnan(zsrc[y, x]), (x, y)


@pytest.mark.parametrize("w,h,n", [(403, 351, 5), (404, 350, 5), (397, 373, 5), (1001, 601, 1)])
def test_four_pixels_a_thread_equal_one(orc, w, h, n):
    """From 600 000 pixels a launch on a thread takes four pixels of a row: a
    batch of that many against single calls below, and a single call above;
    every remainder of 4 on some level, and borders on all sides."""
    cam = camera(w, h)
    args = (w, h, cam.cx, cam.cy, cam.fx, cam.fy)
    T0, T1, f0, f1 = make_pair(cam, 23)
    filt = RGBDOdometry(*args).bilateral(f1.depth, 5.0)
    odos = [fed(RGBDOdometry(*args), T0, f0, f1, filt) for _ in range(n + 1)]
    odos[0].getIncrementalTransformation(T0[:3, 3], T0[:3, :3], False, 10.0, True, False, False)
    for o in odos[1:]:
        o.set_pose(T0[:3, 3], T0[:3, :3])
    Batch(odos[1:]).track(False, 10.0, True, False, False)
    assert w * h * n >= 600_000 > (w * h if n > 1 else 0)
    for level in range(3):
        a, m = odos[0].read_buffer("dxy", level), odos[0].read_buffer("zsrc", level)
        for o in odos[1:]:
            assert np.array_equal(a, o.read_buffer("dxy", level)), level
            assert np.array_equal(m.view(np.uint32), o.read_buffer("zsrc", level).view(np.uint32)), level
    check_level(odos[0].read_buffer("next_image", 2).astype(np.int32), odos[0].read_buffer("next_depth", 2), a, m, 2)


@pytest.mark.parametrize("w,h", [(640, 624), (736, 712), (1280, 960)])
def test_so3_of_many_pixels_a_thread(orc, w, h):
    """Levels 2 of 24 960, 32 752 and 76 800 pixels over 8 192 threads: the
    call is the oracle's, one launch or one per iteration."""
    cam = camera(w, h)
    args = (w, h, cam.cx, cam.cy, cam.fx, cam.fy)
    T0, T1, f0, f1 = make_pair(cam, 22)
    filt = RGBDOdometry(*args).bilateral(f1.depth, 5.0)
    out = []
    for spin in (1 << 20, -1):
        odo = fed(RGBDOdometry(*args), T0, f0, f1, filt)
        odo.set_so3_loop(spin)
        out.append(pose_of(*odo.getIncrementalTransformation(T0[:3, 3], T0[:3, :3], False, 10.0, True, False, True)))
    assert np.array_equal(out[0], out[1])
    ref = fed(orc.Odometry(*args), T0, f0, f1, filt)
    exp = pose_of(*ref.getIncrementalTransformation(T0[:3, 3], T0[:3, :3], False, 10.0, True, False, True))
    dt, dr = synth.pose_error(out[0], exp)
    assert dt <= 1e-3 and dr <= 0.1, (dt, dr)
