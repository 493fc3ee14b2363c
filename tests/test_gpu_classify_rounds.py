"""The set-up of the cut pass over more band cells than its work-groups hold at once: with 1024
work-groups of 64 cells a round, 84^3 cells to cut (nine rounds and a part) fill a work-group's
buffer of 512 in the eighth, so that it is emptied once in mid-run and once at the end; 44^3 cells
(two rounds) at the end only. A checkerboard of full and empty cells, all of them band cells with
the other phase upstream: every cell must reach the cut list exactly once, and VF matches the
oracle's.

Tolerance: the same operations but for the order of a cell's leaf sums, 1e-12 of the cell as in the
other transport tests.
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


@pytest.mark.parametrize("n", [44, 84])
def test_every_cell_of_a_wide_band_is_cut(mist, oracle, n):
    param, _ = W.deformation3d(n)
    out = []
    for cls in (mist.Context, oracle.OracleContext):
        c = cls(param)
        rng = np.random.default_rng(n)
        v = c.get("VF")
        c.set("VF", np.indices(v.shape).sum(0) % 2 + 0.0)
        c.vof_init()
        u = c.get("uf")
        c.set("uf", rng.uniform(0.4, 1.0, (1, *u.shape[1:])) * np.where(rng.random((1, *u.shape[1:])) < 0.5, -1, 1)
              + np.zeros_like(u))
        for f in ("vf", "wf"):
            c.set(f, np.zeros_like(c.get(f)))
        before = W.interior(c.mesh, c.get("VF"), vof=True).copy()
        assert np.abs(W.interior(c.mesh, c.get("band"))).max() == 0
        c.transport(0.2 / n)
        out.append(W.interior(c.mesh, c.get("VF"), vof=True))
    assert (out[1] != before).mean() > 0.95
    assert np.abs(out[0] - out[1]).max() <= 1e-12
