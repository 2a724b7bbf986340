"""The frame loop's components on streams of their own (surfel_set_stream and
splat_set_stream on the loop's handles): poses, model and prediction are those
of a loop that stays on the odometry's stream, bit for bit, wherever the
streams are moved and for host and device frames."""
import ctypes

import numpy as np
import pytest

from slam_amd import splat, surfels, synth
from slam_amd.frame_loop import FrameLoop, LoopParams, lib
from slam_amd.odometry import _check, _p

pytestmark = pytest.mark.gpu


def prediction(handle, w, h):
    out = {}
    for which, (ch, dt) in splat._SHAPE.items():
        out[which] = np.zeros((h, w, ch), dt)
        _check("splat_read", splat.lib().splat_read(handle, which, _p(out[which])))
    return out


def handles(loop):
    sp, m = ctypes.c_void_p(), ctypes.c_void_p()
    _check("efloop_get_handles", lib().efloop_get_handles(loop._h, None, ctypes.byref(sp), ctypes.byref(m)))
    return sp, m


@pytest.mark.parametrize("device", [False, True])
@pytest.mark.parametrize("moved,at", [("model", 1), ("prediction", 1), ("both", 0), ("both", 2)])
def test_components_on_streams_of_their_own(moved, at, device):
    import torch
    cam = synth.CAM_320
    scene = synth.Scene(17)
    poses = synth.spline_trajectory(6, seed=17, max_step_m=0.01, max_step_deg=0.5)
    frames = [scene.render(T, cam, noise_seed=k, model=False) for k, T in enumerate(poses)]
    args = (cam.width, cam.height, cam.cx, cam.cy, cam.fx, cam.fy)
    plain, loop = (FrameLoop(*args, LoopParams(max_surfels=400_000)) for _ in range(2))
    streams = [torch.cuda.Stream() for _ in range(2)]
    sp, model = handles(loop)
    for k, f in enumerate(frames):
        if k == at:
            if moved != "prediction":
                _check("surfel_set_stream", surfels.lib().surfel_set_stream(model, streams[0].cuda_stream))
            if moved != "model":
                _check("splat_set_stream", splat.lib().splat_set_stream(sp, streams[1].cuda_stream))
        rgb, depth = (torch.from_numpy(a).cuda() for a in (f.rgb, f.depth)) if device else (f.rgb, f.depth)
        torch.cuda.synchronize()
        assert np.array_equal(plain.process(rgb, depth), loop.process(rgb, depth)), k
        a, b = (prediction(q, cam.width, cam.height) for q in (handles(plain)[0], sp))
        for which in a:
            assert np.array_equal(a[which].view(np.uint8), b[which].view(np.uint8)), (k, which)
    a, b = plain.model.model(), loop.model.model()
    assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
