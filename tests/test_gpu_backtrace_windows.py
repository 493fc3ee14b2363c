"""The back-trace and the index boxes from coordinates loaded around a vertex and a cell: points that
stay within a cell of their start, points one cell away and points beyond the loaded coordinates
(several cells) end where the oracle's walks end, so that VF after one step is the oracle's.

Tolerance: the stages are the same operations in the same order; VF as in the transport tests, 1e-12.
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


@pytest.mark.parametrize("scheme", ["RK4", "Euler", "Midpoint"])
@pytest.mark.parametrize("shift", [0.4, 1.3, 2.6])  # cells a step carries a point
@pytest.mark.parametrize("dims,per", [((16, 13, 15), ""), ((17, 16, 14), "xyz")])
def test_carried_sphere_matches_oracle(mist, oracle, dims, per, shift, scheme):
    param, _ = W.deformation3d(dims[0], Ny=dims[1], Nz=dims[2], CFL=3.0, projection_method=scheme, xper="x" in per,
                               yper="y" in per, zper="z" in per)
    out = []
    for cls in (mist.Context, oracle.OracleContext):
        c = cls(param)
        c.init_vof("sphere", 0.21, 0.47, 0.52, 0.49)
        c.vof_init()
        for n, s, a in (("uf", 1.0, 0), ("vf", -0.8, 1), ("wf", 0.6, 2)):
            f = c.get(n)
            wave = np.sin(2 * np.pi * np.arange(f.shape[(a + 1) % 3]) / dims[(a + 1) % 3])
            shape = [1, 1, 1]
            shape[(a + 1) % 3] = -1
            c.set(n, s * (1.0 + 0.2 * wave.reshape(shape)) + np.zeros_like(f))
        c.transport(shift / dims[0])
        out.append(W.interior(c.mesh, c.get("VF"), vof=True))
    assert np.abs(out[0] - out[1]).max() <= 1e-12
