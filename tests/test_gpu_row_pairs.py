"""The fused row launch that transforms two rows at a time: row counts that leave part of the last
work item empty, both row plans of every small length, and fields of very different size."""

import numpy as np
import pytest

import mhdflows_amd as M
from mhdflows_amd import ic
from oracle.integrator import rel_l2
from oracle.rhs import calcN as o_calcN
from test_gpu_parity import _calcN_gpu, _resample, pair, say

pytestmark = pytest.mark.gpu


# rows (ny * nz) against 2 * 128 / (nx / values a thread) rows a work item: less than one, one and
# a remainder, a whole number
@pytest.mark.parametrize("shape", [(8, 8, 8), (8, 24, 8), (16, 8, 24), (24, 8, 16), (32, 8, 48), (48, 16, 8), (64, 8, 8),
                                   (96, 8, 24), (128, 24, 8), (1024, 8, 8)])
@pytest.mark.parametrize("T", [np.float64, np.float32])
@pytest.mark.parametrize("physics", ["MHD", "HD"])
def test_rhs_every_plan_and_remainder(shape, T, physics):
    if shape[0] == 24 and T == np.float64 and physics == "MHD":
        pytest.skip("refused: 24-point rows in Float64 MHD")
    if shape[0] > 128 and T == np.float32:
        pytest.skip("Float32 rounding grows with the largest wavenumber: test_large_lengths_each_axis has the bound")
    say("row pairs", shape, T.__name__, physics)
    nx, ny, nz = shape
    mhd = physics == "MHD"
    fields = _resample(ic.solenoidal_modes(5, k0=2.0, kmax=min(shape) / 3 - 0.5, mhd=mhd), nx, ny, nz, mhd)
    for var in (0, 1):
        o, p = pair(nx, ny=ny, nz=nz, T=T, physics=physics, fields=fields)
        M.variants(p, [-1, -1, -1, -1, var])
        N_ref = np.zeros_like(o.sol)
        N_gpu, _ = _calcN_gpu(p, o.sol.copy())
        o_calcN(N_ref, o.sol.copy(), 0.0, o)
        assert rel_l2(N_gpu, N_ref) < (1e-12 if T == np.float64 else 2e-5), var


@pytest.mark.parametrize("n", [32, 96])
def test_small_magnetic_field_keeps_its_accuracy(n):
    """A seed magnetic field of 1e-6 next to velocities of order one: the induction part of a Float32
    right-hand side is as close to the Float64 oracle, relative to itself, as for fields of one size."""
    say("seed field", n)
    o64, _ = pair(n, T=np.float64, kmax=n / 4.0)
    fields = [np.array(v) * (1.0 if f < 3 else 1e-6) for f, v in enumerate(o64.vars)]
    o64, _ = pair(n, T=np.float64, fields=fields)
    o32, p = pair(n, T=np.float32, fields=[f.astype(np.float32) for f in fields])
    N_ref = np.zeros_like(o64.sol)
    o_calcN(N_ref, o64.sol.copy(), 0.0, o64)
    N_gpu, _ = _calcN_gpu(p, o32.sol.copy())
    for f in (slice(0, 3), slice(3, 6)):
        assert rel_l2(N_gpu[f], N_ref[f]) < 2e-5


# the long lengths with a factor 3, where some threads sit passes out; the Float32 bound of 128 points
# grows with the largest wavenumber, which multiplies the products' rounding
@pytest.mark.parametrize("nx", [192, 384, 768])
@pytest.mark.parametrize("T", [np.float64, np.float32])
@pytest.mark.parametrize("physics", ["MHD", "HD"])
def test_rhs_long_rows_with_a_factor_3(nx, T, physics):
    say("long rows", nx, T.__name__, physics)
    mhd = physics == "MHD"
    fields = _resample(ic.solenoidal_modes(6, k0=2.0, kmax=2.1, mhd=mhd), nx, 8, 24, mhd)
    for var in (0, 1):
        o, p = pair(nx, ny=8, nz=24, T=T, physics=physics, fields=fields)
        M.variants(p, [-1, -1, -1, -1, var])
        N_ref = np.zeros_like(o.sol)
        N_gpu, _ = _calcN_gpu(p, o.sol.copy())
        o_calcN(N_ref, o.sol.copy(), 0.0, o)
        assert rel_l2(N_gpu, N_ref) < (1e-12 if T == np.float64 else 2e-5 * nx / 128), var
