"""The kernel profile and the stage times of a step: every pass of the loop is counted, the plane
constants' among them although they are made with the normals."""
import numpy as np
import pytest

from ns_multiphase_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [12, 1])  # a periodic axis of one cell keeps the separate pass
def test_step_counts_the_plane_constants(nz):
    from ns_multiphase_amd import solver
    param, ic = W.deformation3d(16, Nz=nz, Lz=nz / 16, zper=nz == 1)
    c = solver.Context(param)
    c.init_vof("circle", 0.2, 0.5, 0.5) if nz == 1 else c.init_vof("sphere", 0.2, 0.5, 0.5, 0.4)
    c.vof_init()
    c.profile(True)
    t = 0.0
    for _ in range(3):
        t, _ = c.vof_step(t)
    prof = c.profile_read()
    cells = int(np.prod(c.mesh.cell_shape()))
    assert prof["plic"][1:] == (3, 3 * cells)
    assert prof["elvira"][1] == 3 and prof["elvira"][2] > 0
    c.compute_plic()
    assert c.profile_read()["plic"][1:] == (4, 4 * cells)
