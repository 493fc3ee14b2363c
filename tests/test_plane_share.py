"""The closed-form liquid share ELVIRA scores its candidates with (PlaneShare, compiled for the
host): against exact rational corner volumes, and against the reference's computePLIC2VF
arithmetic on a cell's 27 neighbours, whose deviation the near-tie test of k_elvira bounds.

Tolerances: a share is a handful of roundings of numbers at most 1, 1e-15 of the exact value; a
neighbour's deviation is the reference's sub-tet determinants' own, which lose the digits of
|x| / h: below share_deviation, the bound k_elvira uses, 3e-15 (N + 1)."""
import ctypes
import os
import shutil
import subprocess
from fractions import Fraction

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "share_harness.hip")
LIB = os.path.join(HERE, "_build", "libshareh.so")


@pytest.fixture(scope="module")
def H():
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    os.makedirs(os.path.dirname(LIB), exist_ok=True)
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-w",
                    SRC, "-o", LIB], check=True, capture_output=True)
    L = ctypes.CDLL(LIB)
    L.h_share.restype = ctypes.c_double
    L.h_share.argtypes = [ctypes.c_void_p, ctypes.c_double]
    L.h_deviation.restype = ctypes.c_double
    L.h_deviation.argtypes = [ctypes.c_double, ctypes.c_double]
    L.h_neighbours.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_double, ctypes.c_void_p]
    return L


def exact_share(m, a):
    """Volume of {m.x < a} in the unit cube, m sorted and positive, by inclusion and exclusion."""
    s = Fraction(0)
    for q in range(8):
        t = a - sum(m[d] for d in range(3) if q >> d & 1)
        if t > 0:
            s += (-1) ** bin(q).count("1") * t ** 3
    return s / (6 * m[0] * m[1] * m[2])


@pytest.mark.parametrize("small", [1.0, 1e-3, 1e-8, 1e-14])
def test_share_against_exact_volumes(H, small):
    rng = np.random.default_rng(7)
    for trial in range(300):
        m = rng.uniform(0.05, 1.0, 3)
        m[trial % 3] *= small
        if trial % 5 == 0:
            m[(trial + 1) % 3] *= small
        m /= m.sum()
        s = np.sort(m)
        # offsets across every part: around each break and its mirror image, the ends, anywhere
        offs = np.concatenate([s, [s[0] + s[1], 0.5], s * (1 - 1e-9), s * (1 + 1e-9), rng.uniform(0, 1, 6), [-0.1, 1.1]])
        for a in np.concatenate([offs, 1 - offs]):
            F = [Fraction(float(v)) for v in s]
            tot = sum(F)
            e = exact_share(F, Fraction(float(a)) * tot)  # the floats' sum is 1 to rounding
            got = H.h_share(m.ctypes.data, float(a))
            assert abs(got - float(min(max(e, Fraction(0)), Fraction(1)))) <= 1e-15, (m, a, got, float(e))


def test_zero_components(H):
    for m, a, v in (((0, 0, 1), 0.3, 0.3), ((0, 1, 0), 0.75, 0.75), ((0, 0.5, 0.5), 0.25, 0.125),
                    ((0.5, 0, 0.5), 0.75, 0.875), ((0.25, 0.75, 0), 0.5, 0.5)):
        mm = np.array(m, float)
        assert abs(H.h_share(mm.ctypes.data, a) - v) <= 1e-15


@pytest.mark.parametrize("N", [(32, 32, 32), (128, 128, 128), (256, 256, 256), (44, 37, 52), (100, 61, 9)])
def test_neighbours_against_reference_arithmetic(H, N):
    rng = np.random.default_rng(N[0])
    n_ = np.array(N, np.int32)
    worst = 0.0
    for trial in range(2000):
        c = np.array([rng.integers(1, v - 2) for v in N], np.int32)
        n = rng.standard_normal(3)
        if trial % 3 == 0:
            n[rng.integers(0, 3)] *= 1e-6
        if trial % 7 == 0:
            n[rng.integers(0, 3)] = 0.0
        n /= np.linalg.norm(n)
        pt = (c + rng.random(3)) / n_
        out = np.zeros(54)
        H.h_neighbours(n_.ctypes.data, c.ctypes.data, n.ctypes.data, float(n @ pt), out.ctypes.data)
        worst = max(worst, np.abs(out[::2] - out[1::2]).max())
    assert worst <= H.h_deviation(1.0, 1.0 / max(N)), worst  # |x| <= 1


@pytest.mark.parametrize("tiny", [1e-99, 1e-101, 1e-155, 1e-200, 1e-309, 5e-324])
def test_vanishing_components(H, tiny):
    """Components whose reciprocals or their products overflow, one at a time and both, at empty and
    full neighbours too: the share is that of a component 0 to rounding, and always a number."""
    for m in ((tiny, 0.3, 0.7), (0.5, tiny, 0.5), (tiny, tiny, 1.0), (tiny, 1.0, 0.0), (0.25, 0.75, tiny)):
        z = [0.0 if v == tiny else v for v in m]
        for a in (-0.5, 0.0, tiny, 0.1, 0.2, 0.5, 0.8, 0.9, 1.0, 1.5):
            got = H.h_share(np.array(m).ctypes.data, a)
            want = H.h_share(np.array(z).ctypes.data, a)
            assert abs(got - want) <= 1e-15, (m, a, got, want)
            assert 0.0 <= want <= 1.0
