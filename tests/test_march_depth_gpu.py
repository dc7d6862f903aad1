"""A depth that nothing compares behind (NaN) ends no ray in any form of the
raymarch: those pixels are the ones without a depth buffer, also where a group
of samples starts in an empty brick and ends in hair."""
import numpy as np
import pytest
import torch

from vkhr_amd import params, synth
from vkhr_amd import device as D

pytestmark = pytest.mark.gpu


# four lanes per pixel at one run and several, one lane over runs, the loop, and the power-of-two form
@pytest.mark.parametrize("w,h,steps", [(96, 80, 128), (97, 82, 300), (400, 302, 101), (200, 300, 40), (520, 400, 256)])
@pytest.mark.parametrize("res", [(40, 33, 50), (90, 100, 120)])
def test_nan_depth_ends_no_ray(device, w, h, steps, res):
    b, vol = D.style_volume(synth.hemisphere_style(700, 12, seed=8), res, device, segments=True)
    sc = synth.make_scene(b, w, h, azimuth_deg=40.0)
    scene = params.camera(sc), params.light(sc), params.strand(b, res), params.render(raycast_steps=float(steps))
    free = D.raymarch(vol, res, *scene, w, h, want_info=True)
    nan = np.random.default_rng(steps).random((h, w)) < 0.5
    depth = np.where(nan, np.nan, 0.0).astype(np.float32)
    out = D.raymarch(vol, res, *scene, w, h, depth_buffer=torch.from_numpy(depth).to(device), want_info=True)
    at = torch.from_numpy(nan).to(device)
    assert int((free["info"][at][:, 0] == 1).sum()) > 500
    assert torch.equal(out["info"][at], free["info"][at])
    assert torch.equal(out["depth"][at], free["depth"][at])
    # (other groups of samples, in another order of float64 sums)
    assert float((out["rgba"][at] - free["rgba"][at]).abs().max()) <= 1.2e-7
