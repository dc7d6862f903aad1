"""Trees, strand orders and bounds on a thread of their own leave the capture
of another thread valid in every mode, the default (global) one included: they
allocate, build in kept memory, wait and free."""
import ctypes as C
import threading

import numpy as np
import pytest
import torch

from tests.test_call_scratch_gpu import BOX, _style
from vkhr_amd import capi
from vkhr_amd import device as D
from vkhr_amd.trace import Bvh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["global", "thread_local", "relaxed"])
@pytest.mark.parametrize("kept", [False, True])
def test_trees_leave_a_capture_valid(device, mode, kept):
    styles = [_style(k, n) for k, n in enumerate((2000, 9000, 2500, 9500))]
    radius = [torch.full((s[0].shape[0],), 0.01, device=device) for s in styles]
    want = [Bvh(s[0], r, s[2]).nodes() for s, r in zip(styles, radius)]
    other, unused = torch.cuda.Stream(), torch.cuda.Stream()
    capi.call("vkhr_release_scratch", other.cuda_stream)
    if kept:
        Bvh(styles[0][0], radius[0], styles[0][2], stream=other)
    x, g, s, errors, trees = torch.zeros(1000, device=device), torch.cuda.CUDAGraph(), torch.cuda.Stream(), [], []
    order = D.sort_strands(styles[1][0], styles[1][2], BOX).cpu().numpy()
    out, box = torch.empty_like(styles[1][2]), capi.make_aabb(BOX)

    def work():
        try:
            for (xyz, _, idx), r in zip(styles, radius):
                Bvh(xyz, r, idx, stream=other)          # freed or kept at once
                trees.append(Bvh(xyz, r, idx, stream=other))
            xyz, _, idx = styles[1]
            capi.call("vkhr_sort_strands", capi.ptr(xyz), xyz.shape[0], capi.ptr(idx), idx.numel(), C.byref(box),
                      capi.ptr(out), capi.stream_of(other))
            capi.call("vkhr_aabb_compute", capi.ptr(xyz), xyz.shape[0], C.byref(capi.AABB()), capi.stream_of(other))
            capi.call("vkhr_release_scratch", unused.cuda_stream)   # the kept memory
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s, capture_error_mode=mode):
        x.add_(1)
        t = threading.Thread(target=work)
        t.start()
        t.join()
        x.add_(1)
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
    assert not errors, errors
    assert float(x[0]) == 6.0 and len(trees) == 4
    assert np.array_equal(out.cpu().numpy(), order)
    for tree, w in zip(trees, want):
        for a, b in zip(tree.nodes(), w):
            assert np.array_equal(a, b)
    capi.call("vkhr_release_scratch", other.cuda_stream)   # (torch hands its streams out again)
