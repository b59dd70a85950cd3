"""Launch choices may change while steps are queued: the graphs being replayed are destroyed only when
their launches have ended, and every queued step runs."""

import numpy as np
import pytest

import mhdflows_amd as M
from mhdflows_amd import ensemble as E
from test_gpu_parity import say

pytestmark = pytest.mark.gpu

NAMES = ("ux", "uy", "uz", "bx", "by", "bz")


def fields(n, seed=0):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((n, n, n)).astype(np.float32) for _ in NAMES]


def test_problem_changes_with_steps_queued():
    say("graph lifetime")
    sols = []
    for wait in (True, False):
        p = M.Problem("MI355X", nx=64, nu=1e-3, eta=1e-3, B_field=True, T=np.float32, dt=1e-4)
        M.SetUpProblemIC(p, *fields(64))
        for k in range(6):
            M.stepforward(p, 41)
            if wait:
                p.sol
            M.row_launch(p, 1 + k % 3)       # plan 1 and its teams: the same bits
            M.stepforward(p, 6)
            if wait:
                p.sol
            M.set_pipeline(p, 1 + k % 2)
        sols.append(p.sol)
    assert np.array_equal(*sols)


def test_group_changes_with_steps_queued():
    say("graph lifetime, groups")
    sols = []
    for wait in (True, False):
        e = E.Ensemble([E.make_config(n, nu=1e-3, eta=1e-3, dt=1e-4) for n in (32, 48, 64)])
        for r, n in enumerate((32, 48, 64)):
            e.set_ic_real(r, fields(n, r))
        e.multi(True)
        for k in range(4):
            e.launch(41)
            if wait:
                e.sync()
            e.multi_classes(k % 2, (k + 1) % 2)
            e.launch(6)
            if wait:
                e.sync()
            e.multi(k % 2 == 0)
        e.sync()
        sols.append([e.get_sol(r) for r in range(3)])
        e.close()
    for a, b in zip(*sols):
        assert np.array_equal(a, b)
