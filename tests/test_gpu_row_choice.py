"""A run ends with the same bits alone and beside others of its grid: the number of runs may choose
another form of the row launch, never another row plan."""

import numpy as np
import pytest

import mhdflows_amd as M
from mhdflows_amd import ensemble as E
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


# grids whose row launch is a team alone and fills the chip with the given number of runs, by rows of
# each plan; one that fills it alone
@pytest.mark.parametrize("shape,many", [((128, 64, 64), 3), ((192, 64, 64), 2), ((256, 32, 32), 8), ((96, 64, 64), 4),
                                        ((128, 96, 96), 2), ((192, 96, 96), 2)])
@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("mhd", [False, True])
def test_alone_and_in_a_group(shape, many, T, mhd):
    say("row choice", shape, many, T.__name__, mhd)
    nx, ny, nz = shape
    names = ("ux", "uy", "uz", "bx", "by", "bz")[:6 if mhd else 3]
    rng = np.random.default_rng(8)
    fields = [rng.standard_normal((nz, ny, nx)).astype(T) for _ in names]
    p = M.Problem("MI355X", nx=nx, ny=ny, nz=nz, nu=1e-3, eta=1e-3, B_field=mhd, T=T, dt=1e-3)
    M.SetUpProblemIC(p, **dict(zip(names, fields)))
    M.stepforward(p, 2)
    for n in (1, many):
        e = E.Ensemble([E.make_config(nx, ny, nz, nu=1e-3, eta=1e-3, T=T, B_field=mhd, dt=1e-3) for _ in range(n)])
        for r in range(n):
            e.set_ic_real(r, fields if r == n - 1 else fields[::-1])
        e.step(2)
        e.sync()
        assert np.array_equal(e.get_sol(n - 1), p.sol), n
        e.close()
