"""The frame loop leaves the cleaned model's count on the device until a call
needs it: the loop's model and counts are those of the same stages called one
by one, each waiting for its count, and its predictions are those of its own
model read back and predicted with the count from the host, bit for bit, also
when the model buffer is full (the device's count then exceeds the surfels
kept)."""
import ctypes

import numpy as np
import pytest
import torch

from slam_amd import splat, synth
from slam_amd.frame_loop import FrameLoop, LoopParams, lib
from slam_amd.odometry import RGBDOdometry, _check, _p
from slam_amd.surfels import SurfelModel

pytestmark = pytest.mark.gpu


def weighting(loop):
    w = ctypes.c_float()
    _check("efloop_get_state", lib().efloop_get_state(loop._h, None, ctypes.byref(w), None))
    return w.value


def check_prediction(loop, pred, p, pose, tick, filt, rgb):
    """The loop's prediction and fill-in against those of its model's copy."""
    sp = ctypes.c_void_p()
    _check("efloop_get_handles", lib().efloop_get_handles(loop._h, None, ctypes.byref(sp), None))
    mine = {}
    for which, (ch, dt) in splat._SHAPE.items():
        mine[which] = np.zeros((pred.height, pred.width, ch), dt)
        _check("splat_read", splat.lib().splat_read(sp, which, _p(mine[which])))
    model = torch.from_numpy(loop.model.model()).cuda()
    torch.cuda.synchronize()
    pred.combinedPredict(pose, model, p.max_depth, p.confidence, tick, tick, p.time_delta)
    pred.fillIn(filt, rgb)
    for which in mine:
        theirs = pred.read(which).reshape(mine[which].shape)
        assert np.array_equal(mine[which].view(np.uint8), theirs.view(np.uint8)), (tick, which)
    assert np.any(mine[splat.FILL_VERTEX][..., 2] > 0)


@pytest.mark.parametrize("w,h,room", [(320, 240, 4.0), (322, 238, 0.5), (97, 81, 0.4)])
def test_loop_model_equals_the_stages_one_by_one(w, h, room):
    cam = synth.Camera(w, h, 0.8 * w, 0.8 * w, w / 2.0, h / 2.0)
    scene = synth.Scene(7)
    poses = synth.spline_trajectory(5, seed=7, max_step_m=0.01, max_step_deg=0.5)
    frames = [scene.render(T, cam, noise_seed=k, model=False) for k, T in enumerate(poses)]
    args = (w, h, cam.cx, cam.cy, cam.fx, cam.fy)
    # (the confidence is that of young surfels, so that the model is predicted)
    p = LoopParams(depth_cutoff=6.0, confidence=0.5, max_surfels=int(room * w * h))
    loop = FrameLoop(*args, p)
    odo, model, pred = RGBDOdometry(*args), SurfelModel(*args, p.max_surfels), splat.IndexMap(*args)
    last_err = 0.0
    for k, f in enumerate(frames):
        pose = loop.process(f.rgb, f.depth)
        filt = odo.bilateral(f.depth, p.depth_cutoff)
        if k == 0:
            model.initialise(f.rgb, f.depth, filt, p.depth_cutoff, 1, p.max_depth)
        elif last_err < 1e-4:
            model.predictIndices(pose, k + 1, p.max_depth, p.time_delta)
            model.fuse(pose, k + 1, f.rgb, f.depth, filt, p.depth_cutoff, p.max_depth, weighting(loop))
            model.predictIndices(pose, k + 1, p.max_depth, p.time_delta)
            model.clean(pose, k + 1, p.confidence, p.time_delta)
        last_err = loop.odo.stats()["lastICPError"] if k else 0.0
        if k == len(frames) - 1 or room < 1:     # read in between, or only at the end
            check_prediction(loop, pred, p, pose, k + 1, filt, f.rgb)
            assert loop.model.lastCount() == model.lastCount() <= p.max_surfels
    a, b = loop.model.model(), model.model()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    if room < 1:
        assert model.lastCount() == p.max_surfels
