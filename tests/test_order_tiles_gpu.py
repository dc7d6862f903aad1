"""vkhr_sort_strands at the sizes where one workgroup runs every stage (4096
pairs) or the stages over the runs (10240 runs of up to 32768 pairs), and the
time of a style of single segments against one of as many launches."""
import time

import pytest
import torch

from tests.test_order_runs_gpu import test_runs_are_sorted_stably as _check
from vkhr_amd import device as D

pytestmark = pytest.mark.gpu

# (pairs, pairs of a run, distinct root positions per axis)
CASES = [(2, 1, 8), (1023, 1, 3), (1025, 1, 1000), (4095, 1, 2), (4096, 4096, 8), (4096, 3, 50), (4097, 2, 50),
         (10237, 1, 1000), (10238, 1, 1), (10240, 1, 1000), (10241, 1, 1000), (10300, 1, 4), (20474, 2, 1000),
         (20480, 2, 1000), (20484, 2, 1000), (32768, 3, 30), (32768, 4, 30), (32768, 1, 1)]


@pytest.mark.parametrize("n,length,spread", CASES)
def test_the_tiles_edges(device, n, length, spread):
    _check(device, n, length, spread)


def test_single_segments_cost_what_strands_do(device):
    """5000 runs of a pair each took a workgroup's attempt, a wait and then
    eleven launches, 105 us, where 1000 pairs took 43; 68 and 39 now."""
    b = dict(origin=(0.0, 0.0, 0.0), size=(1.0, 1.0, 1.0), radius=1.0, volume=1.0)
    took = []
    for n in (5000, 1000):
        xyz = torch.rand(2 * n, 3, device=device)
        idx = torch.arange(2 * n, dtype=torch.int32, device=device)
        best = 1.0
        for _ in range(60):
            torch.cuda.synchronize()
            t = time.perf_counter()
            D.sort_strands(xyz, idx, b)
            best = min(best, time.perf_counter() - t)
        took.append(best)
    assert took[0] <= 2.1 * took[1], took
