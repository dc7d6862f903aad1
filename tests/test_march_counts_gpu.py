"""The raymarch around the sample counts from which step counts off the powers
of two march over runs of equal increments (56 with four lanes per pixel, 96
with one), alone and in a batch, against the float64 oracle; images of an odd
height without their middle row, whose horizontal rays run along a texel plane
(the sign of a 1e-15 weight decides there whether a sample counts as hair)."""
import numpy as np
import pytest
import torch

from tests.parity import compare_raymarch
from vkhr_amd import params, synth
from vkhr_amd import device as D
from vkhr_amd.batch import Batch, StyleBuffers

pytestmark = pytest.mark.gpu
RES = (40, 33, 50)


def _numpy(out):
    return {k: v.cpu().numpy() for k, v in out.items()}


# 800 pixels a step take four lanes: all but the last two sizes
@pytest.mark.parametrize("w,h", [(96, 95), (128, 80), (300, 262), (301, 261)])
@pytest.mark.parametrize("steps", [5, 24, 55, 56, 57, 95, 96, 97])
def test_counts_match_the_oracle(device, steps, w, h):
    b, vol = D.style_volume(synth.hemisphere_style(1500, 12, seed=6), RES, device, segments=True)
    sc = synth.make_scene(b, w, h, azimuth_deg=70.0)
    scene = params.camera(sc), params.light(sc), params.strand(b, RES), params.render(raycast_steps=float(steps))
    host = dict(density=vol["density"].cpu().numpy(), tangents=vol["tangents"].cpu().numpy())
    pixels = np.arange(w * h, dtype=np.int64)
    if h % 2:
        pixels = pixels[pixels // w != h // 2]
    free = _numpy(D.raymarch(vol, RES, *scene, w, h, want_info=True))
    compare_raymarch(free, host, RES, *scene, w, h, pixels=pixels)
    depth = np.where(np.random.default_rng(steps).random((h, w)) < 0.5, 1.0, free["depth"] + 1e-3)
    depth = np.clip(depth, 0.0, 1.0).astype(np.float32)
    out = D.raymarch(vol, RES, *scene, w, h, depth_buffer=torch.from_numpy(depth).to(device), want_info=True)
    # (the oracle takes the depth of the pixels it is given)
    compare_raymarch(_numpy(out), host, RES, *scene, w, h, pixels=pixels, depth_buffer=depth)


def test_a_batch_of_counts(device):
    """Each style's image is the one of its own raymarch (1.2e-7: another form
    may sum in another order)."""
    w, h = 300, 262
    styles = [StyleBuffers(synth.hemisphere_style(800, 12, seed=k), 40, w, h, device, azimuth=30.0 * k,
                           steps=float(steps)) for k, steps in enumerate((24, 95, 96, 97, 128, 300))]
    batch = Batch(styles, w, h)
    for _ in range(2):
        batch.launch()
    torch.cuda.synchronize()
    for s in styles:
        vol = dict(density=s.density, cells=s.cells, tangents=s.tangents, occupancy=s.occupancy)
        one = D.raymarch(vol, (s.n,) * 3, s.cam, s.light, s.sp, s.rp, w, h)["rgba"]
        assert float(one.abs().max()) > 0.1
        assert float((one - s.rgba).abs().max()) <= 1.2e-7
