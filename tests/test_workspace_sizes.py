"""The workspaces that backward asks for and insists on, without a GPU: no larger than they have been for any shape (a caller may
have laid its memory out by them), and without the fp32 partials of dW where the dlogits are kept and one launch stores dW."""
import ctypes as C
import random

import pytest

from slowrun_amd import _lib

# (N, d, V, offsets): smallest, default and kept-mode workspace in bytes with a chunk sum for every 16 entries and one fp32 partial of dW
BEFORE = {
    (65536, 2560, 50304, 1): (810541056, 4348906752, 797627136), (2048, 768, 50304, 1): (237446400, 415660800, 312350720),
    (61, 2560, 50304, 1): (597558784, 597558784, 584644864), (200, 64, 1000, 4): (68574208, 68574208, 68311808),
    (30011, 2560, 50257, 1): (695216896, 2296521216, 682302976), (32768, 1024, 50304, 3): (349046272, 2061443328, 408484096),
    (300, 16, 7, 1): (67616512, 135053056, 134921728), (131072, 256, 256, 4): (150542336, 251410176, 217847552),
    (200000, 64, 512, 1): (143931136, 211449344, 144324096), (16384, 4096, 131072, 1): (2334098432, 4448543744, 2300535808),
    (130000, 2560, 50304, 1): (1020851968, 7981233920, 1524361728), (131072, 1600, 50304, 2): (804870144, 7661979904, 1153452800),
    (256, 4096, 524288, 1): (8796832000, 8796832000, 8662581504)}


@pytest.mark.parametrize("shape", sorted(BEFORE))
def test_no_workspace_has_grown(shape):
    s = _lib.sizes_for(*shape)
    least, default, kept = BEFORE[shape]
    assert s.bwd_workspace_min_bytes <= least and s.bwd_workspace_bytes <= default and s.bwd_workspace_kept_bytes <= kept
    assert s.bwd_workspace_min_bytes <= s.bwd_workspace_bytes


def test_kept_dlogits_need_no_partial_of_dw():
    N, d, V = 65536, 2560, 50304
    s = _lib.sizes_for(N, d, V)
    rows, cols = d, -(-V // 256) * 256
    assert s.bwd_workspace_kept_bytes < BEFORE[N, d, V, 1][2] - rows * cols * 4 + (N // 8 - N // 16 + 1) * (rows * 4 + 8) + 4096
    # beyond the rows of one launch there are partials again
    assert _lib.sizes_for(131073, d, V).bwd_workspace_kept_bytes > _lib.sizes_for(131072, d, V).bwd_workspace_kept_bytes + rows * cols * 4


def test_sums_of_the_shorter_columns_fit_where_the_partials_would_lie():
    """One launch over dlogits formed again: its workspace is that of several launches, which hold a partial of dW and half as many chunk sums."""
    rng = random.Random(5)
    up = lambda n: (n + 255) // 256 * 256
    for _ in range(3000):
        K = rng.choice((1, 1, 2, 4))
        N = round(2 ** rng.uniform(0, 16.5))
        V = round(2 ** rng.uniform(0, 18))
        d = 16 * round(2 ** rng.uniform(0, 9))
        dq, Vp, NE = up(d), up(V), N * K
        sums = lambda slots: up((2 * slots + 2) * 4) + up(slots * dq * 4)
        assert sums(min(NE // 8, V + NE // 256) + 1) <= sums(NE // 16 + 1) + up(dq * Vp * 4), (N, K, d, V)
