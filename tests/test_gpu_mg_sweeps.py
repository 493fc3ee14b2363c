"""The multigrid's smoothing kernels at the sizes where they can go wrong, against the oracle:
after exactly two V-cycles every variant (a launch per colour with two or four planes per thread,
fused sweeps over LDS tiles of both shapes, an odd sweep left over) holds the oracle's iterate.

Tolerance: an FP64 V-cycle is the same sequence of relaxations on both sides, each of which
rounds to a few 1e-16 of the largest correction; two cycles of 40 contracting relaxations per
cell stay below 1e-11 of max|P|. In mixed precision the corrections carry FP32 rounding, 6e-8
per relaxation: 1e-5 of max|P|.
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


# A periodic axis with an odd extent on some level has neighbours of one colour, whose relaxations
# have no defined order: the periodic cases stay even down to their coarsest level (mg_lvl).
CASES = [
    ((40, 24, 16), (10, 10), "", 1),       # one small-tile level, partial tiles
    ((40, 24, 16), (3, 1), "", 1),         # a sweep left over after the pairs
    ((64, 48, 80), (10, 10), "", 1),       # the large tile, then the small one
    ((72, 24, 24), (4, 5), "xz", 3),       # periodic, the last tile of a row cut off
    ((128, 32, 32), (2, 2), "xyz", 1),     # periodic, whole tiles
    ((136, 40, 72), (2, 3), "", 1),        # a launch per colour, two planes per thread, cut-off tiles
    ((160, 64, 32), (1, 1), "yz", 1),
    ((128, 128, 72), (2, 2), "", 1),       # a launch per colour, four planes per thread
]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dims,nu,per,lvl", CASES)
def test_two_vcycles_match_oracle(mist, oracle, dims, nu, per, lvl, precision):
    dt = 1e-3
    p = W.mms_params(dims[0], Ny=dims[1], Nz=dims[2], Ly=dims[1] / dims[0], Lz=dims[2] / dims[0], mg_nu1=nu[0],
                     mg_nu2=nu[1], mg_max_cycles=2, mg_lvl=lvl, xper="x" in per, yper="y" in per, zper="z" in per)
    P = []
    for cls in (mist.Context, oracle.OracleContext):
        c = cls(p)
        W.mms_setup(c, dt)
        c.pressure_solve(dt, 1e-30, precision, check=False)
        P.append(W.interior(c.mesh, c.get("P")))
    scale = np.abs(P[1]).max()
    assert scale > 0
    assert np.abs(P[0] - P[1]).max() <= (1e-11 if precision == "fp64" else 1e-5) * scale


# Every level above the coarsest has even extents, so remainders are two rows or planes short of a
# tile or a single plane; the residual of the outer loop meets any extent on a mesh of one level.
REMAINDERS = [
    ((32, 22, 18), (3, 2), ""),            # LDS tiles cut off along y and z
    ((26, 18, 22), (2, 3), ""),            # and along x; the residual's last planes
    ((13, 11, 7), (2, 2), ""),             # one level: odd extents in the residual
    ((512, 256, 1), (2, 2), ""),           # a plane: one per thread
    ((1024, 1024, 1), (2, 2), ""),         # a plane among the large levels
    ((1024, 512, 2), (2, 1), ""),          # two planes among the large levels
    ((256, 1, 192), (2, 2), ""),           # a plane along x and z
    ((64, 2, 256), (2, 1), "x"),           # a slab: a launch per colour, one plane per thread
    ((64, 64, 64), (2, 1), ""),            # 256 LDS tiles, the most that take them
    ((64, 64, 72), (2, 1), ""),            # 288
    ((128, 128, 2), (2, 2), ""),           # a slab in 256 small LDS tiles
]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dims,nu,per", REMAINDERS)
def test_two_vcycles_with_remainders_match_oracle(mist, oracle, dims, nu, per, precision):
    test_two_vcycles_match_oracle(mist, oracle, dims, nu, per, 1, precision)


# Rows shorter than a wave of pairs keep plain order above the levels of the LDS sweeps. The longest
# side is 1 here: cells of a whole or half a wavelength would leave no right-hand side.
SHORT_ROWS = [
    ((1, 256, 192), (2, 2), ""),           # rows of one cell
    ((2, 512, 384), (2, 2), ""),
    ((16, 256, 128), (2, 1), "yz"),        # plain order, then the LDS tiles
    ((56, 96, 64), (1, 2), ""),            # below the least length of a split row, and at it
    ((64, 96, 64), (1, 2), ""),
    ((16, 512, 1), (2, 2), ""),
]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dims,nu,per", SHORT_ROWS)
def test_two_vcycles_of_short_rows_match_oracle(mist, oracle, dims, nu, per, precision):
    L = [d / max(dims) for d in dims]
    p = W.mms_params(dims[0], Ny=dims[1], Nz=dims[2], Lx=L[0], Ly=L[1], Lz=L[2], mg_nu1=nu[0], mg_nu2=nu[1],
                     mg_max_cycles=2, mg_lvl=1, xper="x" in per, yper="y" in per, zper="z" in per)
    P = []
    for cls in (mist.Context, oracle.OracleContext):
        c = cls(p)
        W.mms_setup(c, 1e-3)
        assert c.pressure_solve(1e-3, 1e-30, precision, check=False)[0] == 2
        P.append(W.interior(c.mesh, c.get("P")))
    scale = np.abs(P[1]).max()
    assert scale > 0.1
    assert np.abs(P[0] - P[1]).max() <= (1e-11 if precision == "fp64" else 1e-5) * scale
