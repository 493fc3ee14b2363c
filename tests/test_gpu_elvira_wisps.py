"""ELVIRA where column sums differ by next to nothing: fields of empty, full and half cells with wisps of
1e-99 down to the smallest double, whose candidate normals have components of that size. No candidate may
be lost to an overflowing reciprocal: the normals are those the oracle keeps.

Tolerance: the device's error of a candidate is exact to rounding and near ties are decided in the
reference's arithmetic, so the same candidate is kept; its components are the same operations, 1e-12.
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


@pytest.mark.parametrize("wisp", [1e-99, 1e-155, 1e-200, 1e-309, 5e-324])
def test_normals_beside_wisps_match_oracle(mist, oracle, wisp):
    n = 24
    param, _ = W.deformation3d(n)
    out = []
    for cls in (mist.Context, oracle.OracleContext):
        c = cls(param)
        rng = np.random.default_rng(3)
        v = c.get("VF")
        v[...] = 0.0
        # single part-filled cells three apart, each with a few wisps around it
        for i in range(6, v.shape[0] - 6, 3):
            for j in range(6, v.shape[1] - 6, 3):
                for k in range(6, v.shape[2] - 6, 3):
                    block = v[i - 1:i + 2, j - 1:j + 2, k - 1:k + 2]
                    block[...] = np.where(rng.random(block.shape) < 0.15, wisp * rng.integers(1, 4), 0.0)
                    block[1, 1, 1] = rng.uniform(0.1, 0.9)
        c.set("VF", v)
        c.compute_normal()
        out.append([W.interior(c.mesh, c.get(a)) for a in ("nx", "ny", "nz")])
    assert np.abs(np.stack(out[1])).max() > 0.5
    for a, b in zip(*out):
        assert np.abs(a - b).max() <= 1e-12
