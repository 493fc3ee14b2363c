"""One transport step whose pre-images grow from a box of two cells per axis to boxes beyond four:
the first cut pass, the wide pass with either order of its sums, and the general walk all take
cells, and VF matches the oracle.

Tolerance: a cell's two volumes are sums of at most 6144 leaf volumes whose sizes add up to a few
cell volumes, each leaf good to some 1e-15 of the cell: 1e-12 of the cell bounds the share.
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


CASES = [((16, 16, 16), 0.01, ""), ((16, 16, 16), 0.04, ""), ((16, 16, 16), 0.08, ""), ((15, 18, 13), 0.1, "xz"),
         ((16, 14, 1), 0.06, "z"), ((14, 17, 16), 0.13, "xyz")]


@pytest.mark.parametrize("dims,dt,per", CASES)
def test_cut_passes_match_oracle(mist, oracle, dims, dt, per):
    param, _ = W.deformation3d(dims[0], Ny=dims[1], Nz=dims[2], Lz=1.0 if dims[2] > 1 else 1.0 / dims[0], CFL=4.0,
                               xper="x" in per, yper="y" in per, zper="z" in per)
    state = []
    for cls in (mist.Context, oracle.OracleContext):
        c = cls(param)
        shape = ("sphere", 0.3, 0.47, 0.52, 0.5) if dims[2] > 1 else ("circle", 0.3, 0.47, 0.52)
        c.init_vof(*shape)
        c.vof_init()
        rng = np.random.default_rng(5)
        for n in ("uf", "vf", "wf"):  # a shear plus noise: neighbouring corners part
            f = c.get(n)
            i, j, k = np.meshgrid(*[np.arange(s) for s in f.shape], indexing="ij")
            q = {"uf": j / dims[1], "vf": k / max(dims[2], 2), "wf": i / dims[0]}[n]
            amp = 0.0 if dims[2] == 1 and n == "wf" else 1.0
            c.set(n, amp * (np.sin(2 * np.pi * q) + 0.3 * rng.standard_normal(f.shape)))
        c.transport(dt)
        state.append(W.interior(c.mesh, c.get("VF"), vof=True))
    assert np.isfinite(state[1]).all()
    assert np.abs(state[0] - state[1]).max() <= 1e-12
