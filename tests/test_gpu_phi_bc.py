"""Boundary planes of the level-set field, written by one launch: the inlet
and outlet columns and the extrapolations below and above, where the columns'
and the planes' threads end on and off a block's 64."""
import numpy as np
import pytest

from tpls_amd.case import Case
from tpls_amd.config import CaseParams
from tpls_amd.initial import make_initial

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nx,ny,nz", [(64, 16, 63), (62, 8, 64), (63, 6, 65), (8, 4, 6), (130, 10, 7)])
def test_boundary_planes(nx, ny, nz, precision):
    p = CaseParams(nx=nx, ny=ny, nz=nz, Re=150.0, mu_plus=2.0, dt=1e-4, noise=1e-2, seed=nx + nz, mom_u=2, mom_v=2,
                   mom_w=2, height=0.47)
    with Case(p, precision=precision, diagnostics=False) as c:
        c.load(*make_initial(p))
        c.step(2)
        phi = c.field("phi2")
    t = np.float64 if precision == "fp64" else np.float32
    phi = phi[:, 1:-1].astype(t)
    L, n = nx + 1, nz + 1
    k = np.arange(1, n)
    z = (k - 0.5) / nz - 0.47
    # z of the order of one: at most three roundings of it
    assert np.abs(phi[0, :, 1:n] - z).max() <= 3 * np.finfo(t).eps
    assert np.array_equal(phi[L, :, 1:n], phi[L - 1, :, 1:n])
    # one rounding each, whether fused or not: twice a value is exact
    assert np.array_equal(phi[:, :, 0], t(2) * phi[:, :, 1] - phi[:, :, 2])
    assert np.array_equal(phi[:, :, n], t(2) * phi[:, :, n - 1] - phi[:, :, n - 2])
