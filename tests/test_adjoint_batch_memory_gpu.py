"""The batched adjoint writes its density gradient with plain stores, whichever
scatter its renders take: it may lie in pinned host memory, where float atomics
of the device would be lost."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from tests.test_adjoint_scatter_gpu import DIFF, _scene, _volume
from vkhr_amd import device as D
from vkhr_amd.adjoint_batch import AdjointBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [(64,), (8,), (64, 8, 64)])   # windows, cells, both
def test_gradient_in_host_memory(device, steps):
    res, w, h = (24, 20, 27), 130, 121
    _, _, b, vol = _volume(res, device, 3)
    prob = SimpleNamespace(width=w, height=h, res=res, diff=D.diff_params(*map(float, DIFF)), vol=lambda s: vol)
    n = res[0] * res[1] * res[2]
    host, got = torch.empty(n, pin_memory=True), []
    for where in (torch.empty(n, device=device), host):
        where.fill_(5.0)
        prob.styles, prob.renders = [dict(d_density=where, d_params=torch.zeros(3, device=device))], []
        for k, s in enumerate(steps):
            cam, light, sp, rp = _scene(b, res, w, h, s)
            target = torch.rand((h, w, 4), generator=torch.Generator().manual_seed(k)).to(device)
            rgba, rec = D.raymarch_record(vol, res, cam, light, sp, rp, prob.diff, w, h)
            prob.renders.append(dict(style=0, cam=cam, light=light, sp=sp, rp=rp, target=target, rgba=rgba,
                                     record=rec, loss=torch.zeros(1, device=device)))
        batch = AdjointBatch(prob)
        batch.launch()
        batch.launch()
        torch.cuda.synchronize()
        got.append(where.cpu().double().numpy().copy())
    assert np.linalg.norm(got[0]) > 0.0
    assert np.linalg.norm(got[1] - got[0]) <= 1e-5 * np.linalg.norm(got[0])   # the order of float32 sums
