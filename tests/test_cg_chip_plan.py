"""The partition of a grid for the on-chip CG (cg_chip_plan), on the host."""
import random

from tests.test_gpu_cg_chip import GRIDS
from tpls_amd import _lib


def test_tested_grids_take_every_segment_length():
    plans = [_lib.test_chip_plan(*g) for g in GRIDS]
    assert plans[-1] is None and all(plans[:-1])
    assert {p[0] for p in plans[:-1]} == {1, 2, 4, 8, 16, 24}


def test_plans_hold_their_grid():
    """Any grid with a plan has a cell of a thread for each of its own, at most
    256 boxes, and the wavefronts that gather 64 boxes each."""
    rng = random.Random(1)
    for _ in range(200):
        g = [rng.randint(4, 300), 2 * rng.randint(2, 80), rng.randint(4, 300)]
        p = _lib.test_chip_plan(*g)
        if p is None:
            assert g[0] * g[1] * g[2] > 2300000
            continue
        cells, threads, blocks = p
        assert cells * threads * blocks >= g[0] * g[1] * g[2]
        assert 1 <= blocks <= 256 and threads % 64 == 0 and 64 <= threads <= (1024 if cells <= 8 else 512)
        assert threads // 64 >= (blocks + 63) // 64
