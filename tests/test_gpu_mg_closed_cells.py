"""Cells without an open face (every coefficient underflows to zero): each V-cycle starts from e = 0
there too, so that after three cycles their pressure is the oracle's, on every way of smoothing the
finest level: a launch per colour with one, two and four planes per thread, the LDS sweeps, rows too
short to split.

Tolerance: as for the other smoothing kernels, 1e-11 of max|P| (FP64).
"""
import numpy as np
import pytest

from ns_multiphase_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mist():
    from ns_multiphase_amd import solver
    solver.lib()
    return solver


@pytest.mark.parametrize("dims", [(128, 96, 1), (96, 64, 64), (128, 128, 64), (32, 32, 32), (16, 160, 128)])
@pytest.mark.parametrize("nu", [(1, 1), (2, 1)])
def test_closed_cells_keep_nothing_of_the_cycle_before(mist, oracle, dims, nu):
    L = [d / max(dims) for d in dims]
    p = W.mms_params(dims[0], Ny=dims[1], Nz=dims[2], Lx=L[0], Ly=L[1], Lz=L[2], mg_nu1=nu[0], mg_nu2=nu[1],
                     mg_max_cycles=3, mg_lvl=1)
    dt = 1e-40
    P = []
    for cls in (mist.Context, oracle.OracleContext):
        c = cls(p)
        W.mms_setup(c, 1e-3)
        g = c.mesh.nghost
        lo = [g + d // 3 for d in dims]
        hi = [max(a + 1, a + d // 4) for a, d in zip(lo, dims)]
        for f in ("denx", "deny", "denz"):  # a block behind faces of coefficient dt / (den h^2) = 0
            a = c.get(f)
            a[...] = 1.0
            a[lo[0]:hi[0] + 1, lo[1]:hi[1] + 1, lo[2]:hi[2] + 1] = 1e300
            c.set(f, a)
        for _ in range(2):  # the second solve finds the arrays as the first left them
            c.set("P", np.zeros_like(c.get("P")))
            assert c.pressure_solve(dt, 1e-300, "fp64", check=False)[0] == 3
        P.append(W.interior(c.mesh, c.get("P")))
    scale = np.abs(P[1]).max()
    assert np.isfinite(scale) and scale > 0
    assert np.abs(P[0] - P[1]).max() <= 1e-11 * scale
