"""A tuned choice belongs to what was measured: the grid, the number of runs and the form of the row
launch."""

import numpy as np
import pytest

import mhdflows_amd as M
from mhdflows_amd import ensemble as E
from test_gpu_parity import say

pytestmark = pytest.mark.gpu

SHAPE = dict(nx=512, ny=16, nz=8)  # a grid that no other test tunes


def problem(T=np.float32):
    return M.Problem("MI355X", **SHAPE, nu=1e-3, eta=1e-3, B_field=True, T=T, dt=1e-3)


def fields(T=np.float32):
    rng = np.random.default_rng(2)
    return {k: rng.standard_normal((8, 16, 512)).astype(T) for k in ("ux", "uy", "uz", "bx", "by", "bz")}


def test_a_set_variant_holds_for_both_forms_of_the_row_launch():
    say("tuned: set")
    p = problem()
    M.variants(p, [-1, -1, -1, -1, 3])
    M.SetUpN97(p)
    assert M.variants(p)[4] == 3
    M.set_forcing(p, 0, 0.0, 0.0)
    assert M.variants(p)[4] == 3


@pytest.mark.parametrize("T", [np.float32, np.float64])
def test_a_tuned_row_launch_stays_with_its_form(T):
    """Tuning with and without a module: each form keeps its own number, in this problem and in
    later ones of the process."""
    say("tuned: forms", T.__name__)
    p = problem(T)
    M.SetUpProblemIC(p, **fields(T))
    M.autotune(p, 2)
    plain = M.variants(p)
    M.SetUpN97(p)
    assert M.variants(p)[4] == 0          # xrow_kernel was not measured yet
    M.autotune(p, 2)
    forced = M.variants(p)[4]
    M.set_forcing(p, 0, 0.0, 0.0)
    assert M.variants(p)[4] == plain[4]
    q = problem(T)
    assert M.variants(q)[4] == plain[4]
    M.SetUpN97(q)
    assert M.variants(q)[4] == forced


def test_a_group_does_not_take_a_single_runs_choice():
    """Single runs tuned to each variant number leave a group's bits alone."""
    say("tuned: groups")
    f = list(fields().values())

    def group():
        e = E.Ensemble([E.make_config(512, 16, 8, nu=1e-3, eta=1e-3, dt=1e-3) for _ in range(3)])
        for r in range(3):
            e.set_ic_real(r, f)
        e.step(2)
        e.sync()
        s = e.get_sol(1)
        e.close()
        return s

    before = group()
    p = problem()
    M.SetUpProblemIC(p, *f)
    M.autotune(p, 2)
    assert np.array_equal(group(), before)
