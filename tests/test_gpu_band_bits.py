"""computeBand! from words of 64 cells: rows of 1, 63, 64, 65 and 130 cells, planes and rows that end
inside a work-group, walls and periodic axes in turn (thinner than the ghost layers among them),
over fields whose phases touch everywhere. The band and all its ghost cells are whole numbers and
equal the oracle's.
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


CASES = [((1, 9, 4), ""), ((1, 5, 6), "x"), ((63, 7, 5), "x"), ((64, 4, 9), "yz"), ((65, 11, 3), "xyz"),
         ((130, 3, 2), "x"), ((64, 9, 1), "z"), ((70, 2, 1), "yz"), ((20, 33, 17), "")]


@pytest.mark.parametrize("dims,per", CASES)
@pytest.mark.parametrize("share", [0.02, 0.5])
def test_band_words_match_oracle(mist, oracle, dims, per, share):
    param, _ = W.deformation3d(16, Nx=dims[0], Ny=dims[1], Nz=dims[2], xper="x" in per, yper="y" in per,
                               zper="z" in per)
    ctx = [mist.Context(param), oracle.OracleContext(param)]
    for seed in range(3):  # a second and a third call also find the ghosts of the one before
        rng = np.random.default_rng(seed)
        v = ctx[0].get("VF")
        full = (rng.random(v.shape) < share).astype(float)
        v = np.where(rng.random(v.shape) < 0.01, rng.random(v.shape), full)
        for c in ctx:
            c.set("VF", v)
            c.compute_band()
        assert np.array_equal(ctx[0].get("band"), ctx[1].get("band"))
