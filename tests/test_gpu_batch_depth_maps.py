"""A batch whose current maps all come from depth images reads their z planes
alone; with one pair from given maps among them it reads the maps whole.  Both
give a pair the same bits, also for sizes that leave a part of a tile."""
import numpy as np
import pytest

from slam_amd import synth
from slam_amd.odometry import Batch, RGBDOdometry

from helpers import CUTOFF, make_pair

pytestmark = pytest.mark.gpu

SIZES = [(320, 240), (97, 81), (211, 160)]


def handle(w, h, seed, maps):
    cam = synth.Camera(w, h, 0.82 * w, 0.82 * w, w / 2.0, h / 2.0)
    T0, T1, f0, f1 = make_pair(cam, seed)
    odo = RGBDOdometry(w, h, cam.cx, cam.cy, cam.fx, cam.fy)
    odo.initFirstRGB(f0.rgb)
    odo.initICPModel(f0.vert4, f0.norm4, CUTOFF, T0.astype(np.float32))
    odo.initRGBModel(f0.rgba)
    if maps:
        odo.initICPMaps(f1.vert4, f1.norm4, CUTOFF)
    else:
        odo.initICPRaw(f1.depth, 5.0, CUTOFF)
    odo.initRGB(f1.rgb)
    odo.set_pose(T0[:3, 3], T0[:3, :3])
    return odo


@pytest.mark.parametrize("icp_weight", [10.0, 100.0])
def test_pairs_do_not_depend_on_what_the_others_read(icp_weight):
    poses = []
    for extra in (False, True):
        odos = [handle(w, h, 31 + i, False) for i, (w, h) in enumerate(SIZES)]
        if extra:
            odos.append(handle(160, 120, 40, True))
        b = Batch(odos)
        b.set_blocks(0)                  # a pair's blocks do not depend on the others
        b.track(False, icp_weight, True, False, False)
        poses.append([np.concatenate([np.ravel(x) for x in o.get_pose()]) for o in odos[:len(SIZES)]])
    for a, b in zip(*poses):
        assert np.array_equal(a, b) and np.isfinite(a).all()


@pytest.mark.parametrize("icp_weight,vga", [(10.0, 2), (100.0, 27)])
def test_z_planes_of_large_launches(icp_weight, vga):
    """The z planes are read from 300 000 pixels a launch (8 million without
    the photometric loads): batches whose finest level, and whose others not,
    reach them, against the same with a pair from maps among them."""
    sizes = [(640, 480)] * vga + [(203, 177), (322, 239)]
    pairs = {}
    poses = []
    for extra in (False, True):
        odos = []
        for w, h in sizes:
            cam = synth.Camera(w, h, 0.82 * w, 0.82 * w, w / 2.0, h / 2.0)
            if (w, h) not in pairs:
                pairs[w, h] = make_pair(cam, 60)
            T0, T1, f0, f1 = pairs[w, h]
            odo = RGBDOdometry(w, h, cam.cx, cam.cy, cam.fx, cam.fy)
            odo.initFirstRGB(f0.rgb)
            odo.initICPModel(f0.vert4, f0.norm4, CUTOFF, T0.astype(np.float32))
            odo.initRGBModel(f0.rgba)
            odo.initICPRaw(f1.depth, 5.0, CUTOFF)
            odo.initRGB(f1.rgb)
            odo.set_pose(T0[:3, 3], T0[:3, :3])
            odos.append(odo)
        assert sum(w * h for w, h in sizes) >= (300_000 if icp_weight < 100 else 8_000_000)
        if extra:
            odos.append(handle(160, 120, 61, True))
        b = Batch(odos)
        b.set_blocks(0)                  # a pair's blocks do not depend on the others
        b.track(False, icp_weight, True, False, False)
        poses.append([np.concatenate([np.ravel(x) for x in o.get_pose()]) for o in odos[:len(sizes)]])
        b.close()
        for o in odos:
            o.close()
    for a, b in zip(*poses):
        assert np.array_equal(a, b) and np.isfinite(a).all()


def test_a_handle_may_change_from_depth_to_maps_and_back():
    odo = handle(211, 160, 50, False)
    b = Batch([odo])
    b.set_graph(True)
    cam = synth.Camera(211, 160, 0.82 * 211, 0.82 * 211, 211 / 2.0, 80.0)
    T0, _, _, f1 = make_pair(cam, 50)
    for maps in (False, True, False):
        if maps:
            odo.initICPMaps(f1.vert4, f1.norm4, CUTOFF)
        else:
            odo.initICPRaw(f1.depth, 5.0, CUTOFF)
        odo.set_pose(T0[:3, 3], T0[:3, :3])
        b.track(False, 100.0, True, False, False)
        new = handle(211, 160, 50, maps)
        Batch([new]).track(False, 100.0, True, False, False)
        assert all(np.array_equal(x, y) for x, y in zip(odo.get_pose(), new.get_pose())), maps
