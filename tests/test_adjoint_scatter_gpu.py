"""The two scatters of the adjoint's primary rays -- windows of texels in LDS
and the cells -- on either side of the rule that picks one (the pixels' pitch
and the step in texels, a wave's box), alone and mixed in one batch, against
the float64 oracle; and an image of few pixels over a large volume costs no
more than one of many."""
import time
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from oracle import raymarch as OR
from vkhr_amd import params, synth
from vkhr_amd import device as D
from vkhr_amd.adjoint_batch import AdjointBatch

pytestmark = pytest.mark.gpu

DIFF = np.array([0.3, 11.0, 80.0], np.float32)


def _volume(res, device, seed=0):
    rng = np.random.default_rng(seed)
    n = res[0] * res[1] * res[2]
    dens = np.where(rng.random(n) < 0.2, rng.random(n), 0.0).astype(np.float32)
    tan = rng.integers(-127, 128, (n, 4)).astype(np.int8)
    b = dict(origin=np.array([-1.0, -0.4, -0.7], np.float32), size=np.array([2.0, 1.5, 1.8], np.float32))
    b["radius"] = np.float32(np.linalg.norm(b["size"]))
    b["volume"] = np.float32(np.prod(b["size"]))
    vol = dict(density_f32=torch.from_numpy(dens).to(device), tangents=torch.from_numpy(tan.reshape(-1)).to(device))
    return dens, tan, b, vol


def _scene(b, res, w, h, steps, away=1.8):
    sc = synth.make_scene(b, w, h, azimuth_deg=33.0, distance_scale=away)
    return params.camera(sc), params.light(sc), params.strand(b, res), params.render(raycast_steps=float(steps))


def _check(gd, gp, dd, dp):
    # float32 sums of float32 products, a few roundings of 6e-8 each, from a
    # float32 image and record
    got = gd.double().cpu().numpy()
    assert np.linalg.norm(got - dd) <= 1e-5 * np.linalg.norm(dd)
    assert np.abs(got - dd).max() <= 1e-4 * np.abs(dd).max()
    assert np.allclose(gp.double().cpu().numpy(), dp, rtol=1e-3, atol=1e-4 * np.abs(dp).max())


# pitch of the pixels in texels: 24^3 at 130 pixels 0.27, at 240 0.15; steps of 1.0 and 3.9 texels; 40^3 at 90 pixels 0.6
@pytest.mark.parametrize("n,w,steps", [(24, 130, 64), (24, 131, 50), (24, 240, 64), (24, 130, 40), (24, 130, 16),
                                       (40, 90, 100), (40, 90, 400), (40, 33, 70)])
def test_either_scatter_matches_the_oracle(device, n, w, steps):
    res, h = (n, n - 3, n + 2), w - 7
    dens, tan, b, vol = _volume(res, device)
    scene = _scene(b, res, w, h, steps)
    diff = D.diff_params(*map(float, DIFF))
    _, rec = D.raymarch_record(vol, res, *scene, diff, w, h)
    g = np.random.default_rng(1).normal(size=(h, w, 4)).astype(np.float32)
    gd, gp = D.raymarch_adjoint(vol, res, *scene, diff, w, h, rec, torch.from_numpy(g).to(device))
    _, dd, dp = OR.raymarch_grad(tan, dens, res, *scene, DIFF, w, h, d_rgba=g.reshape(-1, 4))
    _check(gd, gp, dd, dp)


@pytest.mark.parametrize("views", [[(64, 1.8)], [(64, 6.0)], [(8, 1.8), (64, 1.8), (64, 6.0), (70, 2.0), (9, 3.0)]])
def test_a_batch_of_both_matches_the_oracle(device, views):
    res, w, h = (24, 20, 27), 130, 121
    dens, tan, b, vol = _volume(res, device, 3)
    prob = SimpleNamespace(width=w, height=h, res=res, diff=D.diff_params(*map(float, DIFF)), vol=lambda s: vol)
    gd, gp = torch.full((res[0] * res[1] * res[2],), 7.0, device=device), torch.full((3,), 7.0, device=device)
    prob.styles, prob.renders = [dict(d_density=gd, d_params=gp)], []
    for k, (steps, away) in enumerate(views):
        cam, light, sp, rp = _scene(b, res, w, h, steps, away)
        target = torch.rand((h, w, 4), generator=torch.Generator().manual_seed(k)).to(device)
        rgba, rec = D.raymarch_record(vol, res, cam, light, sp, rp, prob.diff, w, h)
        prob.renders.append(dict(style=0, cam=cam, light=light, sp=sp, rp=rp, target=target, rgba=rgba, record=rec,
                                 loss=torch.zeros(1, device=device)))
    batch = AdjointBatch(prob)
    for _ in range(3):   # overwritten by each launch
        batch.launch()
    torch.cuda.synchronize()
    dd, dp = 0.0, 0.0
    for r in prob.renders:
        g = (2.0 * (r["rgba"] - r["target"])).cpu().numpy()
        _, d, p = OR.raymarch_grad(tan, dens, res, r["cam"], r["light"], r["sp"], r["rp"], DIFF, w, h,
                                   d_rgba=g.reshape(-1, 4))
        dd, dp = dd + d, dp + p
    _check(gd, gp, dd, dp)


@pytest.mark.parametrize("n", [128, 200])
def test_few_pixels_cost_no_more_than_many(device, n):
    """Windows over few, far-apart rays took 1.05 ms at 64^2 pixels of 128^3
    (3.9 of 200^3) where 512^2 pixels took a fifth of that."""
    res = (n, n, n)
    _, _, b, vol = _volume(res, device)
    vol["density_f32"] *= 0.02
    diff = D.diff_params(*map(float, DIFF))
    grads = torch.zeros(n ** 3, device=device), torch.zeros(3, device=device)
    took = []
    for w in (64, 512):
        scene = _scene(b, res, w, w, 64)
        rgba, rec = D.raymarch_record(vol, res, *scene, diff, w, w)
        best = 1.0
        for _ in range(20):
            torch.cuda.synchronize()
            t = time.perf_counter()
            D.raymarch_adjoint(vol, res, *scene, diff, w, w, rec, rgba, *grads)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t)
        took.append(best)
    assert took[0] <= took[1], took
