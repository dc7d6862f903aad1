"""A tree of over 2^28 segments: every launch of its build holds all of them,
so that rays find the last segments given and those whose codes sort last.
Takes about 110 GB of device memory (skipped where there is less)."""
import numpy as np
import pytest
import torch

from vkhr_amd.trace import Bvh

pytestmark = pytest.mark.gpu

SIDE = 1448          # distinct segments in a grid of columns along z
LAST = 4096          # given once, after the repeated ones


def test_the_last_segments_are_found(device):
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 150 << 30:
        pytest.skip("needs 150 GB of free device memory")
    u, n = SIDE * SIDE, (1 << 28) + LAST
    g = np.random.default_rng(0)
    at = np.arange(u)
    a = np.stack([at % SIDE, at // SIDE, SIDE * g.random(u)], 1) / SIDE
    k = np.arange(LAST)
    b = np.stack([(20 * (k % 64) + 3.0), (20 * (k // 64) + 7.5), np.full(LAST, 2.0 * SIDE)], 1) / SIDE
    start = np.concatenate([a, b])
    xyz = np.empty((2 * len(start), 3), np.float32)
    xyz[0::2], xyz[1::2] = start, start + [0.3 / SIDE, 0.0, 0.0]
    seg = torch.arange(n, dtype=torch.int32, device=device)
    seg[: n - LAST] %= u
    seg[n - LAST:] -= n - LAST - u
    idx = torch.empty(2 * n, dtype=torch.int32, device=device)
    idx[0::2], idx[1::2] = 2 * seg, 2 * seg + 1
    del seg
    torch.cuda.empty_cache()
    tree = Bvh(torch.from_numpy(xyz).to(device), torch.full((len(xyz),), 1e-5, device=device), idx)
    pick = np.concatenate([g.integers(0, u, 4096), [0, u - 1]])   # the first of a segment's repetitions is the closest's tie
    target = np.concatenate([a[pick], b])
    rays = np.zeros((len(target), 8), np.float32)
    rays[:, :2] = target[:, :2] + [0.15 / SIDE, 0.0]
    rays[:, 2], rays[:, 6], rays[:, 7] = -1.0, 1.0, 10.0
    _, _, hit = tree.trace_rays(torch.from_numpy(rays).to(device))
    want = np.concatenate([pick, n - LAST + k])
    assert np.array_equal(hit.cpu().numpy(), want)
    del tree, idx
    torch.cuda.empty_cache()
