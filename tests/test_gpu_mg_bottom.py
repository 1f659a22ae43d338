"""The bottom of the V-cycle in one block: hierarchies whose first level there
is the largest one taken, just past it, one pair wide in a direction, and with
a coarsest level of many cells.  The cycle evaluates the oracle's operations in
the oracle's order without FMA contraction: a few ulps (1e-13 normwise)."""
import numpy as np
import pytest

from oracle import binding as B
from tests.compare import relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nu", [1, 2, 3])
@pytest.mark.parametrize("nx,ny,nz", [
    (64, 16, 32),      # 4096, 512, 64 cells
    (72, 32, 32),      # 36x16x16 = 9216 cells: that level runs in many blocks, the next in one
    (64, 32, 32),      # 32x16x16 = 8192: in FP64 past what the LDS holds, in FP32 not
    (72, 32, 16),      # 36x16x8 = 4608, about the most in FP64
    (128, 8, 16), (8, 64, 8), (8, 8, 128),
    (176, 48, 80),     # coarsest 22x6x10 alone
    (48, 48, 48),      # coarsest 6x6x6 below 1728 cells
    (272, 8, 16),      # coarsest 68x2x4: its tables stay outside LDS
    (544, 8, 16)])     # coarsest 136x2x4: longer than the tables go, by sweeps
def test_vcycle_matches_oracle(nx, ny, nz, nu):
    from tpls_amd import _lib
    c = (3.0, 1.0, 2.0)
    r = np.random.default_rng(nx + ny + nz + nu).standard_normal(nx * ny * nz)
    z_o, nl_o = B.mg_apply(r, nx, ny, nz, *c, 2 * sum(c), nu)
    z_g, nl_g = _lib.test_mg_apply(r, nx, ny, nz, *c, 2 * sum(c), nu)
    assert nl_o == nl_g
    assert relerr(z_g, z_o) < 1e-13


@pytest.mark.parametrize("mode", [1, 2])
def test_grouped_cycle_equals_alone(mode):
    """FP32 and FP64 cycles whose bottoms start on different levels (FP32 takes about twice the cells)."""
    from tpls_amd.case import Case, batch_step, set_batch_grouped
    from tpls_amd.config import CaseParams
    from tpls_amd.initial import make_initial
    spec = [((64, 32, 64), "fp32"), ((64, 32, 64), "fp64"), ((96, 24, 48), "fp32"), ((64, 16, 32), "fp64"),
            ((32, 8, 16), "fp32"), ((64, 32, 32), "fp32"), ((64, 32, 32), "fp64")]
    ps = [CaseParams(nx=n[0], ny=n[1], nz=n[2], Re=200.0, mu_plus=3.0, seed=q, noise=1e-2, ksp_pc="mg")
          for q, (n, _) in enumerate(spec)]

    def make():
        cs = [Case(p, precision=t) for p, (_, t) in zip(ps, spec)]
        for c, p in zip(cs, ps):
            c.load(*make_initial(p))
        return cs

    alone, batch = make(), make()
    for c in alone:
        c.step(2)
    set_batch_grouped(mode)
    try:
        batch_step(batch, 2)
    finally:
        set_batch_grouped(1)
    for a, b in zip(alone, batch):
        assert a.diag() == b.diag()
        for f in ("u2", "v2", "w2", "pres"):
            assert np.array_equal(a.field(f), b.field(f))
