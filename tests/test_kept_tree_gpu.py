"""The device keeps the memory of the last tree destroyed, whatever it kept
before: a small tree's memory does not stand in a large one's place, nor a
large one's in that of small ones."""
import numpy as np
import pytest
import torch

from tests.test_call_scratch_gpu import _style
from vkhr_amd import capi
from vkhr_amd.trace import Bvh

pytestmark = pytest.mark.gpu


def _given_back():
    """Bytes that a release on a stream without scratch frees: the kept memory."""
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    capi.call("vkhr_release_scratch", torch.cuda.Stream().cuda_stream)
    return torch.cuda.mem_get_info()[0] - before


@pytest.mark.parametrize("sizes", [(100, 90000), (90000, 100, 90000), (100, 3000, 90000)])
def test_the_last_tree_is_kept(device, sizes):
    styles = {n: _style(n, n) for n in set(sizes)}
    radius = {n: torch.full((s[0].shape[0],), 0.01, device=device) for n, s in styles.items()}
    _given_back()
    for n in sizes:
        Bvh(styles[n][0], radius[n], styles[n][2])     # built, then destroyed at once
    pairs = styles[sizes[-1]][2].numel() // 2
    assert _given_back() >= 100 * pairs                # a tree is over 128 bytes a pair
    assert _given_back() < 100 * pairs                 # (once)


def test_trees_in_turn_are_the_same(device):
    a, b = _style(1, 400), _style(2, 60000)
    r = [torch.full((s[0].shape[0],), 0.01, device=device) for s in (a, b)]
    want = [Bvh(a[0], r[0], a[2]).nodes(), Bvh(b[0], r[1], b[2]).nodes()]
    for _ in range(4):
        for s, q, w in zip((a, b), r, want):
            for x, y in zip(Bvh(s[0], q, s[2]).nodes(), w):
                assert np.array_equal(x, y)
