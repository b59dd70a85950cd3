"""Float32 right-hand sides of flows that do not vary along one axis, under a strong mean field, a mean
flow or a jet along that axis: the components across it do not see it (its flux has k = 0 along the
axis), so they stay as accurate as without it.  Compared on the kept modes: two rows transformed as one
complex row round differently, so a flow independent of y gets a difference between even and odd rows,
which is the mode k_y = ny/2, and every user of a right-hand side discards it.
"""

import numpy as np
import pytest

import mhdflows_amd as M
from oracle.grid import dealias_
from oracle.integrator import rel_l2
from oracle.rhs import calcN as o_calcN
from test_gpu_parity import _calcN_gpu, pair, say

pytestmark = pytest.mark.gpu

ALONG = {"mean 100": (100.0, 1.0), "mean 1e4": (1e4, 1.0), "jet 100": (0.0, 100.0)}  # mean, rms


def plane_flow(n, axis, rng, mean, jet):
    """Three components [c][z][y][x] independent of x (axis 0), y or z: a solenoidal flow of rms 1 across
    the axis, mean + jet * (rms 1) along it."""
    k = np.fft.fftfreq(n, 1.0 / n)
    q, p = np.meshgrid(k, k, indexing="ij")
    shape = np.exp(-(p * p + q * q) / 18.0) * (np.maximum(abs(p), abs(q)) < n / 3 - 1)
    psi, w = (np.fft.fft2(rng.standard_normal((n, n))) * shape for _ in range(2))
    first, second, w = (np.fft.ifft2(a).real for a in (1j * q * psi, -1j * p * psi, w))
    rms = np.sqrt(np.mean(first ** 2 + second ** 2) / 2)
    across = [a for a in (0, 1, 2) if a != axis]
    out = [None] * 3
    # the array's first index is the slower of the two axes across (z before y before x)
    out[across[0]], out[across[1]] = first / rms, second / rms
    out[axis] = mean + jet * w / np.sqrt(np.mean(w ** 2))
    return [np.ascontiguousarray(np.broadcast_to(np.expand_dims(f, 2 - axis), (n, n, n))) for f in out]


# 32^3, and 96^3 in both row plans and with a wave per product: every row launch of a right-hand side
@pytest.mark.parametrize("n,var", [(32, 0), (96, 0), (96, 1), (96, 2)])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("physics,field", [("MHD", "b"), ("MHD", "u"), ("HD", "u")])
@pytest.mark.parametrize("along", list(ALONG))
def test_components_across_a_strong_field(n, var, axis, physics, field, along):
    say("guide field", n, var, "xyz"[axis], physics, field, along)
    rng = np.random.default_rng(17)
    mhd = physics == "MHD"
    strong, weak = ALONG[along], (0.0, 1.0)
    fields = plane_flow(n, axis, rng, *(strong if field == "u" else weak))
    if mhd:
        fields += plane_flow(n, axis, rng, *(strong if field == "b" else weak))
    o32, p = pair(n, T=np.float32, physics=physics, fields=[f.astype(np.float32) for f in fields])
    o64, _ = pair(n, T=np.float64, physics=physics, fields=fields)
    M.variants(p, [-1, -1, -1, -1, var])
    sol = o32.sol.copy()
    N_ref = np.zeros_like(o64.sol)
    o_calcN(N_ref, sol.astype(np.complex128), 0.0, o64)
    N_gpu, _ = _calcN_gpu(p, sol)
    for N, o in ((N_ref, o64), (N_gpu, o32)):
        dealias_(N, o.grid)
    across = [a for a in (0, 1, 2) if a != axis]
    # the bound of a Float32 right-hand side of these sizes
    assert rel_l2(N_gpu[across], N_ref[across]) < 2e-5
