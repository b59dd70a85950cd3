"""The spectral launch's two access forms (by the size of the state of all runs) give the same bits: a
few runs of a grid against the same runs among many."""

import numpy as np
import pytest

from mhdflows_amd import ensemble as E
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stepper", ["RK4", "LSRK54"])
@pytest.mark.parametrize("mhd,many", [(True, 20), (False, 40)])   # 64^3: 29 MB a run, 14 MB without b
def test_few_and_many_runs_agree(stepper, mhd, many):
    say("spectral forms", stepper, mhd)
    rng = np.random.default_rng(4)
    fields = [rng.standard_normal((64, 64, 64)).astype(np.float32) for _ in range(6 if mhd else 3)]
    sols = []
    for n in (2, many):
        e = E.Ensemble([E.make_config(64, nu=1e-3, eta=1e-3, B_field=mhd, stepper=stepper, dt=1e-3) for _ in range(n)])
        e.multi(False)
        for r in (0, 1):
            e.set_ic_real(r, fields if r == 0 else fields[::-1])
        e.step(3)
        e.sync()
        sols.append([e.get_sol(0), e.get_sol(1)])
        e.close()
    for a, b in zip(*sols):
        assert np.array_equal(a, b)
