"""The frame loop leaves the cleaned model's count on the device until a call
needs it: the loop's model, counts and predictions are those of the same
stages called one by one, each waiting for its count, also when the model
buffer is full (the device's count then exceeds the surfels kept)."""
import numpy as np
import pytest

from slam_amd import splat, synth
from slam_amd.frame_loop import FrameLoop, LoopParams
from slam_amd.odometry import RGBDOdometry
from slam_amd.surfels import SurfelModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,room", [(320, 240, 4.0), (322, 238, 0.5), (97, 81, 0.4)])
def test_loop_model_equals_the_stages_one_by_one(w, h, room):
    cam = synth.Camera(w, h, 0.8 * w, 0.8 * w, w / 2.0, h / 2.0)
    scene = synth.Scene(7)
    poses = synth.spline_trajectory(5, seed=7, max_step_m=0.01, max_step_deg=0.5)
    frames = [scene.render(T, cam, noise_seed=k, model=False) for k, T in enumerate(poses)]
    args = (w, h, cam.cx, cam.cy, cam.fx, cam.fy)
    p = LoopParams(depth_cutoff=6.0, max_surfels=int(room * w * h))
    loop = FrameLoop(*args, p)
    odo, model, pred = RGBDOdometry(*args), SurfelModel(*args, p.max_surfels), splat.IndexMap(*args)
    last_err, fill = 0.0, None
    for k, f in enumerate(frames):
        pose = loop.process(f.rgb, f.depth)
        filt = odo.bilateral(f.depth, p.depth_cutoff)
        if k == 0:
            model.initialise(f.rgb, f.depth, filt, p.depth_cutoff, 1, p.max_depth)
        elif last_err < 1e-4:
            d = np.linalg.inv(pose.astype(np.float64)) @ last.astype(np.float64)
            move = max(np.linalg.norm(d[:3, 3]), np.arccos(np.clip((np.trace(d[:3, :3]) - 1) / 2, -1, 1)))
            weight = np.float32(max(np.float32(1) - min(np.float32(move), np.float32(0.01)) / np.float32(0.01), 0.5))
            model.predictIndices(pose, k + 1, p.max_depth, p.time_delta)
            model.fuse(pose, k + 1, f.rgb, f.depth, filt, p.depth_cutoff, p.max_depth, float(weight))
            model.predictIndices(pose, k + 1, p.max_depth, p.time_delta)
            model.clean(pose, k + 1, p.confidence, p.time_delta)
        last_err = loop.odo.stats()["lastICPError"] if k else 0.0
        last = pose.copy()
        if k == len(frames) - 1 or room < 1:     # read in between, or only at the end
            assert loop.model.lastCount() == model.lastCount() <= p.max_surfels
    a, b = loop.model.model(), model.model()
    assert a.shape == b.shape
    # the weighting's rotation angle is formed by other means here: positions to 1e-4
    assert np.nanmax(np.abs(a[:, :3] - b[:, :3])) < 1e-4
    if room < 1:
        assert model.lastCount() == p.max_surfels
