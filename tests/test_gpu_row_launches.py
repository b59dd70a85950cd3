"""Every row launch of a right-hand side against the oracle, asked for by itself: both row plans and
both teams, whatever the choice for the grid would be."""

import numpy as np
import pytest

import mhdflows_amd as M
from mhdflows_amd import ic
from oracle.integrator import rel_l2
from oracle.rhs import calcN as o_calcN
from test_gpu_parity import _calcN_gpu, _resample, pair, say

pytestmark = pytest.mark.gpu


# row counts (ny * nz) that leave part of the last work item empty, fill it, or are less than one; the
# Float32 bound of 128 points grows with the largest wavenumber
@pytest.mark.parametrize("shape", [(8, 8, 24), (16, 24, 8), (24, 8, 16), (32, 8, 48), (48, 16, 8), (64, 24, 8), (96, 8, 24),
                                   (128, 24, 8), (192, 8, 24), (256, 24, 8), (384, 8, 8), (512, 8, 24), (768, 8, 8),
                                   (1024, 8, 8)])
@pytest.mark.parametrize("T", [np.float64, np.float32])
@pytest.mark.parametrize("physics", ["MHD", "HD"])
def test_each_launch_against_the_oracle(shape, T, physics):
    nx, ny, nz = shape
    if nx == 24 and T == np.float64 and physics == "MHD":
        pytest.skip("refused: 24-point rows in Float64 MHD")
    say("row launches", shape, T.__name__, physics)
    mhd = physics == "MHD"
    fields = _resample(ic.solenoidal_modes(9, k0=2.0, kmax=min(shape) / 3 - 0.5, mhd=mhd), nx, ny, nz, mhd)
    o, p = pair(nx, ny=ny, nz=nz, T=T, physics=physics, fields=fields)
    N_ref = np.zeros_like(o.sol)
    o_calcN(N_ref, o.sol.copy(), 0.0, o)
    for launch in (0, 1, 2, 3) if nx <= 256 else (0, 1):
        assert M.row_launch(p, launch) == launch
        N_gpu, _ = _calcN_gpu(p, o.sol.copy())
        assert rel_l2(N_gpu, N_ref) < (1e-12 if T == np.float64 else 2e-5 * max(1, nx / 128)), launch


def test_what_sets_and_ends_a_launch():
    p = M.Problem("MI355X", nx=64, B_field=True, T=np.float32, dt=1e-3)
    assert M.row_launch(p) == 2                                       # the choice for a 64^3 run
    assert M.row_launch(p, 0) == 0 and M.variants(p)[4] == 0
    M.variants(p, [-1, -1, -1, -1, 1])
    assert M.row_launch(p) == 1
    for bad in (4, 7):
        with pytest.raises(M.MHDError):
            M.row_launch(p, bad)
    q = M.Problem("MI355X", nx=512, ny=8, nz=8, B_field=True, T=np.float32, dt=1e-3)
    with pytest.raises(M.MHDError):
        M.row_launch(q, 2)
    M.SetUpN97(p)
    assert M.row_launch(p) == -1
    with pytest.raises(M.MHDError):
        M.row_launch(p, 1)


# 768-point Float64 rows are 1.8 times as slow with the six values a thread of plan 1
@pytest.mark.parametrize("nx,T,mhd,launch", [(768, np.float64, True, 0), (768, np.float64, False, 0),
                                             (768, np.float32, True, 1), (512, np.float32, True, 0)])
def test_choice_for_long_rows(nx, T, mhd, launch):
    p = M.Problem("MI355X", nx=nx, ny=64, nz=64, B_field=mhd, T=T, dt=1e-3)
    assert M.row_launch(p) == launch
