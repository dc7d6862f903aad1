"""The index and tangent generators at the mean strand lengths where the lanes
per strand change, against numpy bit for bit (the same float32 operations in
the same order), and their time on strands of two vertices."""
import time

import numpy as np
import pytest
import torch

from vkhr_amd import device as D
from vkhr_amd.capi import call, ptr, stream_of

pytestmark = pytest.mark.gpu


# all of one length; and a mean that one long strand or many short ones set
@pytest.mark.parametrize("lengths", [[k] * n for k in (1, 2, 3, 4, 5, 8, 9, 10, 16) for n in (1, 300)] +
                         [[2] * 999 + [1500], [1] * 500 + [40] * 20, [3, 700, 3], [1, 1, 1, 2], [40] * 10 + [1] * 2000])
def test_generators_by_mean_length(device, lengths):
    off = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint32)
    v = np.random.default_rng(len(lengths)).normal(size=(int(off[-1]), 3)).astype(np.float32)
    last = np.zeros(len(v), bool)
    last[off[1:] - 1] = True
    k = np.nonzero(~last)[0]
    d = v[k + 1] - v[k]
    q = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]
    tan = np.zeros_like(v)
    tan[k] = d * (np.float32(1.0) / np.sqrt(q))[:, None]
    long = np.asarray(lengths) > 1
    tan[off[1:][long] - 1] = tan[off[1:][long] - 2]
    dv, do = D.to_dev(v, device), D.to_dev(off, device)
    assert np.array_equal(D.generate_indices(do).cpu().numpy().reshape(-1, 2), np.stack([k, k + 1], 1))
    assert np.array_equal(D.generate_tangents(dv, do).cpu().numpy(), tan)


@pytest.mark.parametrize("what", ["tangents", "indices"])
def test_short_strands_cost_no_more(device, what):
    """8M vertices: with 16 lanes for each strand of two 158 us (indices 94),
    in strands of thirteen 63 (30)."""
    took = []
    for strands, length in ((4000000, 2), (615384, 13)):
        off = (torch.arange(strands + 1, device=device) * length).int()
        xyz = torch.rand(strands * length, 3, device=device)
        out = torch.empty(2 * strands * length, 3, device=device)
        best = 1.0
        for _ in range(20):
            torch.cuda.synchronize()
            t = time.perf_counter()
            if what == "tangents":
                call("vkhr_generate_tangents", ptr(xyz), ptr(off), strands, ptr(out), stream_of())
            else:
                call("vkhr_generate_indices", ptr(off), strands, ptr(out), stream_of())
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t)
        took.append(best)
    assert took[0] <= 1.5 * took[1], took
