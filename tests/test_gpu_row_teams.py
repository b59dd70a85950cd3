"""Row launches of small grids: a wave per product (or two) gives the bits of a wave per row pair."""

import math

import numpy as np
import pytest

import mhdflows_amd as M
from oracle.integrator import rel_l2
from test_gpu_parity import say

pytestmark = pytest.mark.gpu

MHD, HD = ("ux", "uy", "uz", "bx", "by", "bz"), ("ux", "uy", "uz")


def problem(shape, T, names, var, seed=1):
    nx, ny, nz = shape
    p = M.Problem("MI355X", nx=nx, ny=ny, nz=nz, nu=1e-3, eta=1e-3, B_field=len(names) == 6, T=T, dt=1e-3)
    M.variants(p, [-1, -1, -1, -1, var])
    rng = np.random.default_rng(seed)
    M.SetUpProblemIC(p, **{k: rng.standard_normal((nz, ny, nx)).astype(T) for k in names})
    return p


# work items of 2 * 64 / (nx / values a thread) rows: a part of one, whole numbers, remainders; the
# time steps depend on the maxima and vars on the full last step
@pytest.mark.parametrize("shape", [(8, 8, 8), (16, 8, 24), (24, 16, 8), (32, 8, 48), (48, 16, 8), (64, 24, 8), (96, 8, 24),
                                   (128, 24, 8), (192, 8, 8), (256, 8, 8)])
@pytest.mark.parametrize("T", [np.float64, np.float32])
@pytest.mark.parametrize("names", [MHD, HD])
def test_teams_give_the_same_bits(shape, T, names):
    if shape[0] == 24 and T == np.float64 and names == MHD:
        pytest.skip("refused: 24-point rows in Float64 MHD")
    say("row teams", shape, T.__name__, len(names))
    if names == HD and shape[0] > 96:
        pytest.skip("a plain launch of these rows uses the other plan")
    out = []
    for var in (1, 0, 2, 3):
        p = problem(shape, T, names, var)
        M.TimeIntegrator(p, math.inf, 2, CFL_Coef=0.3)
        out.append([p.sol.copy(), p.clock.t] + [getattr(p.vars, k) for k in names])
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert np.array_equal(a, b)


# grids past the rule of the teams, with short rows: both plans
@pytest.mark.parametrize("shape", [(8, 384, 512), (16, 256, 384), (24, 256, 192), (32, 192, 256), (64, 128, 192)])
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_short_rows_of_large_grids(shape, T):
    if shape[0] == 24 and T == np.float64:
        pytest.skip("refused: 24-point rows in Float64 MHD")
    say("short rows", shape, T.__name__)
    a, b = (problem(shape, T, MHD, var) for var in (0, 1))
    M.stepforward(a, 2)
    M.stepforward(b, 2)
    assert rel_l2(b.sol, a.sol) < (1e-12 if T == np.float64 else 2e-5)
