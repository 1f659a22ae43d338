"""On small grids each Helmholtz sweep of u, v and w goes out as one launch
(launch_jacobi3, launch_sor3, launch_sor_odd3 or, with
more blocks than CUs, launch_sor_pair3, launch_helmholtz_bc3).  Timing
a kernel class brackets single launches, so a case with the timer on runs one
component at a time: both give the same bits, whatever the tile shapes, the
precision, the periods (tiles with rows left over) and the iteration counts."""
import dataclasses

import numpy as np
import pytest

from tpls_amd.case import Case
from tpls_amd.config import CaseParams
from tpls_amd.initial import make_initial

pytestmark = pytest.mark.gpu

BASE = CaseParams(nx=64, ny=16, nz=24, Re=150.0, mu_plus=3.0, dt=2e-4, noise=1e-2, seed=11, mom_u=8, mom_v=8, mom_w=8)
# tiles, sor_fused: unstaged and staged, every odd pass, 16-row staged tiles
SHAPES = [((1, 1, 4, 8, 8, -1), -1), ((8, 4, 8, 8, 8, -1), -1), ((4, 2, 8, 8, 8, -1), 1),
          ((4, 2, 8, 8, 2, 2), 1), ((4, 2, 4, 8, 4, 4), 1), ((4, 2, 8, 8, 8, 8), 1),
          ((4, 2, 8, 8, 8, 16), -1)]


def fields(p, init, precision, tiles, fused, timed):
    with Case(p, precision=precision, tiles=tiles, sor_fused=fused, diagnostics=False) as c:
        c.load(*init)
        if timed:
            c.time_kernels("advect")
        c.step(3)
        return {f: c.field(f) for f in ("u2", "v2", "w2", "phi2", "pres")}


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nx,ny,nz,mom", [(64, 16, 24, (8, 8, 8)), (30, 8, 9, (8, 6, 4)), (66, 10, 7, (4, 6, 10)),
                                          (150, 46, 33, (6, 6, 6)), (130, 48, 18, (4, 8, 8)), (9, 32, 40, (3, 5, 2)),
                                          (290, 96, 12, (4, 4, 4))])
def test_three_components_in_one_launch(nx, ny, nz, mom, precision):
    p = dataclasses.replace(BASE, nx=nx, ny=ny, nz=nz, mom_u=mom[0], mom_v=mom[1], mom_w=mom[2])
    init = make_initial(p)
    for tiles, fused in SHAPES:
        one = fields(p, init, precision, tiles, fused, True)
        three = fields(p, init, precision, tiles, fused, False)
        for f in one:
            assert np.array_equal(one[f], three[f]), (tiles, fused, f)
    print(f"[three at once] {nx}x{ny}x{nz} {precision} {mom}", flush=True)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_above_the_largest_grid_of_the_three(precision):
    """Past 12 M cells FP64 runs each component's loop whole and FP32 the
    lock-step of launch_sor_pair3, with loops of different lengths."""
    p = dataclasses.replace(BASE, nx=512, ny=128, nz=192, mom_u=8, mom_v=6, mom_w=8, ksp_pc="mg", dt=2e-5)
    init = make_initial(p)
    tiles = (4, 2, 8, 8, 8, 8)
    one = fields(p, init, precision, tiles, 1, True)
    three = fields(p, init, precision, tiles, 1, False)
    for f in one:
        assert np.array_equal(one[f], three[f]), f
