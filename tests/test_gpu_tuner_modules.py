"""The autotuner times what a step runs: negative damping and volume penalisation have one row launch,
which it leaves alone, and the tuned problem still steps as the oracle does."""

import numpy as np
import pytest

import mhdflows_amd as M
from oracle.integrator import rel_l2, run_steps
from test_gpu_parity import say
from test_gpu_vp import vp_pair

pytestmark = pytest.mark.gpu


def row_line(report):
    return [line for line in report.splitlines() if line.startswith("xrow_fused")][0]


@pytest.mark.parametrize("physics", ["MHD", "HD"])
def test_penalised_runs(physics):
    say("tuner vp", physics)
    o, p = vp_pair(physics=physics)
    assert "ms" not in row_line(M.autotune(p, 2))
    run_steps(o, 2)
    M.stepforward(p, 2)
    assert rel_l2(p.sol, o.sol) < 1e-12


def test_negative_damping_and_a_static_force():
    say("tuner nd")
    p = M.Problem("MI355X", nx=32, nu=1e-2, eta=1e-2, B_field=True, T=np.float64, dt=1e-3)
    rng = np.random.default_rng(0)
    M.SetUpProblemIC(p, **{k: rng.standard_normal((32, 32, 32)) for k in ("ux", "uy", "uz", "bx", "by", "bz")})
    f = rng.standard_normal((32, 32, 32))
    M.SetUpND(p, 1.0, f, f, f)
    assert "ms" not in row_line(M.autotune(p, 2))
    M.SetUpN97(p)
    assert "v0=" in row_line(M.autotune(p, 2))
