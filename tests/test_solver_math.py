"""Rounding of the Riemann solver's helpers, on the host (no GPU)."""
import ctypes as C
import os
import subprocess
from fractions import Fraction

import numpy as np
import pytest

from magic_master_amd.build import CSRC, HIPCC

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("solver") / "libsolver.so")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I" + CSRC, "-o", so,
                    os.path.join(HERE, "solver_math.hip")], check=True, stderr=subprocess.DEVNULL)
    return C.CDLL(so)


def _p(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


def _rel(got, exact):
    """Largest relative error, exactly, in units of 2**-53."""
    return max(float(abs(Fraction(g) - e) / abs(e) * 2 ** 53) for g, e in zip(got.tolist(), exact))


@pytest.mark.parametrize("err", [0.0, 2.0 ** -51, 1e-14])   # of the reciprocal: FP64's, the FP32 form's
def test_quotient_from_an_approximate_reciprocal(lib, err):
    """(gamma - 1) / a**2, kinetic energies over rho and the limiters' ratios
    keep the error of one rounding (a unit of 2**-53, and what the residual's
    own rounding can add) though the reciprocal has a larger one."""
    rng = np.random.default_rng(5)
    n = 20000
    num = rng.uniform(0.2, 0.7, n) * 2.0 ** rng.integers(-40, 40, n) * rng.choice([-1, 1], n)
    den = rng.uniform(1.0, 2.0, n) * 2.0 ** rng.integers(-60, 40, n)
    rcp = (1.0 / den) * (1.0 + err * rng.uniform(-1, 1, n))
    out = np.empty(n)
    lib.quotients(_p(num), _p(den), _p(rcp), _p(out), n)
    exact = [Fraction(a) / Fraction(b) for a, b in zip(num.tolist(), den.tolist())]
    assert _rel(out, exact) <= 1.0 + 1e-9
    if err:
        assert _rel(num * rcp, exact) > 1.5        # the product with the reciprocal does not
