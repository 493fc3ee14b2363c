"""The zero-mean gauge of the pressure solve: P less its mean, whose sum is the fixed order of 4096
work-groups of 256 threads on meshes of any size (fewer on small ones). A tolerance that the first
residual meets leaves P itself, so the result is known to the bit: each thread adds the cells it
strides over, a work-group its threads as a tree, and one work-group the partial sums the same way.
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


def _tree(a):
    """Sums over 256 threads (axis 0) as the work-group's tree adds them."""
    while a.shape[0] > 1:
        a = a[: a.shape[0] // 2] + a[a.shape[0] // 2:]
    return a[0]


def _strided(a, threads):
    s = np.zeros(threads)
    for q in range(0, a.size, threads):
        part = a[q:q + threads]
        s[: part.size] += part
    return s


def device_sum(a):
    blocks = min(4096, -(-a.size // 256))
    part = _tree(_strided(a, 256 * blocks).reshape(blocks, 256).T.copy())
    return _tree(_strided(part, 256))


@pytest.mark.parametrize("dims", [(24, 20, 16), (128, 128, 64), (256, 192, 64), (4, 512, 512)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_mean_of_p_is_summed_in_the_fixed_order(mist, dims, precision):
    c = mist.Context(W.mms_params(dims[0], Ny=dims[1], Nz=dims[2], Ly=dims[1] / dims[0], Lz=dims[2] / dims[0]))
    W.mms_setup(c, 1e-3)
    P = c.get("P")
    P[...] = np.random.default_rng(dims[0]).standard_normal(P.shape)
    c.set("P", P)
    cycles, _ = c.pressure_solve(1e-3, 1e300, precision)
    assert cycles == 0
    a = W.interior(c.mesh, P)
    want = a - device_sum(a.ravel(order="F")) / a.size
    assert np.array_equal(W.interior(c.mesh, c.get("P")), want)
