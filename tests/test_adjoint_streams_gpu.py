"""Adjoints of several styles on streams of their own that add to one set of
parameters (one material): no update is lost."""
import numpy as np
import pytest
import torch

from tests.test_adjoint_scatter_gpu import DIFF, _scene, _volume
from vkhr_amd import capi
from vkhr_amd import device as D

pytestmark = pytest.mark.gpu


def test_streams_share_the_parameters(device):
    """Four streams; plain adds of the three sums lost updates here now and
    then, since nothing orders the calls."""
    res, w, h, rounds = (8, 8, 8), 16, 16, 300
    diff = D.diff_params(*map(float, DIFF))
    jobs = []
    for k in range(4):
        _, _, b, vol = _volume(res, device, k)
        scene = _scene(b, res, w, h, 16)
        rgba, rec = D.raymarch_record(vol, res, *scene, diff, w, h)
        one = D.raymarch_adjoint(vol, res, *scene, diff, w, h, rec, rgba)[1].double()
        jobs.append((vol, scene, rgba, rec, torch.zeros(512, device=device), torch.cuda.Stream(), one))
    shared = torch.zeros(3, device=device)
    torch.cuda.synchronize()
    for _ in range(rounds):
        for vol, scene, rgba, rec, d_density, stream, _ in jobs:
            with torch.cuda.stream(stream):
                D.raymarch_adjoint(vol, res, *scene, diff, w, h, rec, rgba, d_density, shared)
    torch.cuda.synchronize()
    want = sum(job[-1] for job in jobs) * rounds
    # 1200 float32 adds, each within 6e-8 of the sum so far; a lost add is about a 1200th
    rel = ((shared.double() - want).abs() / (sum(job[-1].abs() for job in jobs) * rounds)).max()
    assert float(rel) <= 7e-5, (shared, want)
    assert np.isfinite(float(rel))
    for job in jobs:   # (torch hands its streams out again)
        capi.call("vkhr_release_scratch", job[5].cuda_stream)
