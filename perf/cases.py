"""Performance cases of the MI355X MHD framework: the calls that its users' programs make, each with
its inputs (``prepare``), one pass (``run``), the work it cannot do without (``work``) and its values in
64 bits (``exact``).

Kinds of cases:

* ``adv``: ``TimeIntegrator(p, Inf, steps - 1)`` with the CFL time step chosen on the device, from
  seeded solenoidal fields: how a simulation is advanced between two looks at it.
* ``step``: ``stepforward(p, steps)`` with a fixed time step: the call of a per-step host loop.
* ``rhs``: ``calcN`` on device arrays: the right-hand side as an operator, for a caller with a time
  stepper of their own.
* ``forced``: ``TimeIntegrator`` with the N97 forcing module, then ``Diagnostics``: one turn of a
  dynamo run's loop.
* ``ens``: an ensemble of runs of uneven grids, advanced together, each state fetched at the end.
"""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mhdflows.jl_amd"))
import mhdflows_amd as M  # noqa: E402
from mhdflows_amd import ensemble as ME  # noqa: E402

INF = float("inf")
# grid lengths that the framework has transforms for, from the smallest that a run makes sense on
LENGTHS = (16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512, 768)
CFL = 0.3


def _case(kind, n, *, ny=None, nz=None, bits=32, mhd=True, stepper="RK4", steps=1, nu=1e-3, nnu=0, box="cube"):
    return {"kind": kind, "nx": n, "ny": ny or n, "nz": nz or n, "bits": bits, "mhd": mhd, "stepper": stepper,
            "steps": steps, "nu": nu, "nnu": nnu, "box": box}


def _ensemble(per_size, sizes, steps, bits=32, stepper="LSRK54"):
    return {"kind": "ens", "runs": per_size, "sizes": sizes, "steps": steps, "bits": bits, "stepper": stepper}


def listed():
    return [
        # the smallest run, one step a call: a host loop that looks at every step (launches and latency)
        dict(_case("step", 32, nu=1e-2), name="step 32 f32"),
        # a small run advanced on the device, the size most often asked for in a stream of small solves
        dict(_case("adv", 64, stepper="LSRK54", steps=20), name="adv 64 f32 lsrk"),
        # a middling run
        dict(_case("adv", 128, steps=10), name="adv 128 f32"),
        # the headline configuration: 256^3 MHD RK4 in Float32 under the CFL condition
        dict(_case("adv", 256, steps=20), name="adv 256 f32"),
        # large single runs: memory-bound, long transforms; the larger one a single whole step
        dict(_case("adv", 512, steps=3, nu=5e-4), name="adv 512 f32"),
        dict(_case("step", 768, nz=512, steps=1, nu=2e-4, box="dx"), name="step 768x768x512 f32"),
        # double precision, asked for by one solve in ten, with the low-storage stepper and a length 3 * 2^n
        dict(_case("adv", 192, bits=64, stepper="LSRK54", steps=4), name="adv 192 f64 lsrk"),
        # hydrodynamics with hyperviscosity in an elongated box, three different lengths
        dict(_case("adv", 192, ny=96, nz=64, mhd=False, steps=8, nu=1e-6, nnu=2, box="dx"), name="adv hd 192x96x64"),
        # the right-hand side as an operator, every mode of it, in both precisions
        dict(_case("rhs", 128, bits=64), name="rhs 128 f64"),
        dict(_case("rhs", 384, ny=128, nz=192, box="dx"), name="rhs 384x128x192 f32"),
        # a forced dynamo run: the forcing module inside the step, then the diagnostics of the loop
        dict(_case("forced", 96, steps=10, nu=2e-3), name="forced 96 f32"),
        # uneven ensemble: 6 runs each of four small grids, advanced together
        dict(_ensemble(6, "32 48 64 96", 40), name="ensemble 24 runs"),
    ]


def _points(c):
    """Grid points times right-hand sides of one pass, weighted by the width of a value and the fields."""
    stages = 4 if c["stepper"] == "RK4" else 5
    if c["kind"] == "ens":
        return sum(n ** 3 for n in _sizes(c)) * c["steps"] * stages * c["bits"] / 32
    rhs = 1 if c["kind"] == "rhs" else c["steps"] * stages
    return c["nx"] * c["ny"] * c["nz"] * rhs * c["bits"] / 32 * (1.0 if c["mhd"] else 0.6)


MOST_POINTS = 768 * 768 * 512 * 4


def _log_pick(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _length_near(x):
    return min(LENGTHS, key=lambda v: abs(math.log(v / x)))


def draw(rng):
    kind = rng.choice(("adv", "adv", "step", "rhs", "forced", "ens"))
    while True:
        bits = 64 if rng.random() < 0.25 else 32
        stepper = rng.choice(("RK4", "RK4", "LSRK54"))
        if kind == "ens":
            sizes = rng.sample((24, 32, 48, 64, 96, 128), rng.randint(2, 4))
            c = _ensemble(rng.randint(2, 6), " ".join(map(str, sorted(sizes))), rng.randint(10, 40), bits, stepper)
            bad = bits == 64 and 24 in sizes
        else:
            base = _log_pick(rng, 24, 640)
            axes = [_length_near(base * (_log_pick(rng, 0.4, 2.2) if rng.random() < 0.5 else 1)) for _ in range(3)]
            mhd = kind == "forced" or rng.random() < 0.75
            c = _case(kind, axes[0], ny=axes[1], nz=axes[2], bits=bits, mhd=mhd, stepper=stepper,
                      steps=1 if kind in ("step", "rhs") else rng.randint(2, 20), nu=_log_pick(rng, 5e-4, 5e-3),
                      nnu=0, box=rng.choice(("cube", "dx")))
            # the framework refuses rows of 24 points in Float64 MHD; host work of large fields is kept out
            bad = (bits == 64 and mhd and axes[0] == 24) or (kind == "forced" and max(axes) > 256)
            bad = bad or axes[0] * axes[1] * axes[2] * bits // 32 > 512 ** 3  # device memory, in 64 bits too
        if not bad and _points(c) <= MOST_POINTS * 0.8:
            return c


# ---- inputs --------------------------------------------------------------------------------------
def _sizes(c):
    return [int(s) for s in c["sizes"].split() for _ in range(c["runs"])]


def _box(c):
    """Box lengths: 2 pi along every axis, or the same grid spacing along every axis."""
    two_pi = 2 * math.pi
    if c["box"] == "cube":
        return two_pi, two_pi, two_pi
    return two_pi, two_pi * c["ny"] / c["nx"], two_pi * c["nz"] / c["nx"]


def _modes(seed, shape, box, mhd, k0=4.0, kmax=16):
    """Seeded solenoidal initial fields, E(k) ~ k^4 exp(-2 (k / k0)^2), rms 1 a component: sparse
    half-spectrum entries ``(kx, l, m)`` and their values (M, nf) for a grid of ``shape`` (nx, ny, nz)."""
    top = [min(kmax, n // 3 - 1) for n in shape]
    p, q, r = np.meshgrid(*[np.arange(-t, t + 1) for t in top], indexing="ij")
    kv = np.stack([p.ravel(), q.ravel(), r.ravel()], 1)
    first = (kv[:, 0] > 0) | ((kv[:, 0] == 0) & ((kv[:, 1] > 0) | ((kv[:, 1] == 0) & (kv[:, 2] > 0))))
    kv = kv[first & ((kv ** 2).sum(1) <= kmax ** 2)]
    k = kv * (2 * math.pi / np.asarray(box))
    k2 = (k ** 2).sum(1)
    rng = np.random.Generator(np.random.PCG64(seed))
    amp = np.sqrt(k2 * np.exp(-2.0 * k2 / k0 ** 2))
    fields = []
    for _ in range(2 if mhd else 1):
        g = rng.standard_normal((len(kv), 3, 2))
        a = (g[..., 0] + 1j * g[..., 1]) * amp[:, None]
        a = a - k * ((k * a).sum(1) / k2)[:, None]
        fields.append(a * math.sqrt(3.0 / (2.0 * (np.abs(a) ** 2).sum())))
    a = np.concatenate(fields, 1) * float(np.prod(shape))
    own = kv[:, 0] == 0          # the kx = 0 plane holds both members of a conjugate pair
    idx = np.concatenate([kv, -kv[own]]) % np.asarray([1 << 30, shape[1], shape[2]])
    return idx.astype(np.int32), np.concatenate([a, a[own].conj()])


def _wavenumbers(shape, box, device):
    nx, ny, nz = shape
    f = dict(dtype=torch.float64, device=device)
    kx = torch.arange(nx // 2 + 1, **f) * (2 * math.pi / box[0])
    ky = torch.fft.fftfreq(ny, 1.0 / ny, **f) * (2 * math.pi / box[1])
    kz = torch.fft.fftfreq(nz, 1.0 / nz, **f) * (2 * math.pi / box[2])
    return kx[None, None, :], ky[None, :, None], kz[:, None, None]


def _dense_state(c, seed):
    """A developed state for the operator calls: solenoidal noise with E(k) ~ k^(-5/3) beyond k = 3 on
    every mode of the half spectrum, the aliased ones included, as a time stepper's update leaves it."""
    shape, box = (c["nx"], c["ny"], c["nz"]), _box(c)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    T = torch.float32 if c["bits"] == 32 else torch.float64
    k = [x.to(T) for x in _wavenumbers(shape, box, "cuda")]
    k2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    amp = (9.0 + k2) ** (-11.0 / 12.0)
    out = []
    for _ in range(2 if c["mhd"] else 1):
        a = []
        for _ in range(3):
            x = torch.randn(shape[2], shape[1], shape[0], generator=gen, device="cuda", dtype=T)
            a.append(torch.fft.rfftn(x) * amp)
        div = (a[0] * k[0] + a[1] * k[1] + a[2] * k[2]) / torch.where(k2 == 0, torch.ones_like(k2), k2)
        a = [v - div * q for v, q in zip(a, k)]
        # rms 1: mean |x|^2 = sum |X|^2 / N^2, interior kx counted twice
        n = float(np.prod(shape))
        s = sum(float((v.real.double() ** 2 + v.imag.double() ** 2).sum()) for v in a) * 2 / n ** 2
        out += [v * math.sqrt(3.0 / s) for v in a]
    return torch.stack(out)


class _DeviceView:
    """A device array of the framework as torch sees it (no copy)."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": typestr, "version": 2}


def _sol_view(p, bits):
    return torch.as_tensor(_DeviceView(p.device_ptrs()[0], p.sol_shape, "<c8" if bits == 32 else "<c16"), device="cuda")


def _np_type(c):
    return np.float32 if c["bits"] == 32 else np.float64


def _problem(c):
    Lx, Ly, Lz = _box(c)
    more = {"calcF": M.N97ForceDriving} if c["kind"] == "forced" else {}
    return M.Problem("MI355X", nx=c["nx"], ny=c["ny"], nz=c["nz"], Lx=Lx, Ly=Ly, Lz=Lz, nu=c["nu"], eta=c["nu"],
                     nnu=c["nnu"], B_field=c["mhd"], stepper=c["stepper"], T=_np_type(c), dt=_fixed_dt(c), **more)


def _fixed_dt(c):
    """The fixed step of the per-step calls, well inside the CFL bound of fields of order one."""
    return 0.03 * 2 * math.pi / max(c["nx"], c["ny"], c["nz"])


def _run_params(c, seed):
    """Per run of an ensemble: viscosity log-uniform in [1e-3, 1e-2] and the spectrum's peak in [2, 6]."""
    rng = np.random.Generator(np.random.PCG64([seed, 7]))
    return [(float(np.exp(rng.uniform(math.log(1e-3), math.log(1e-2)))), float(rng.uniform(2, 6))) for _ in _sizes(c)]


def prepare(case, seed):
    c = case
    if c["kind"] == "ens":
        params = _run_params(c, seed)
        e = ME.Ensemble([ME.make_config(n, nu=nu, eta=nu, T=_np_type(c), stepper=c["stepper"])
                         for n, (nu, _) in zip(_sizes(c), params)])
        for i, (n, (_, k0)) in enumerate(zip(_sizes(c), params)):
            e.set_ic_modes(i, *_modes(seed * 1000 + i, (n, n, n), (2 * math.pi,) * 3, True, k0))
            e.set_cfl(i, CFL)
        return {"case": c, "e": e}
    p = _problem(c)
    state = {"case": c, "p": p}
    if c["kind"] == "rhs":
        state["sol"] = _dense_state(c, seed)
        state["N"] = torch.empty_like(state["sol"])
        torch.cuda.synchronize()
        return state
    M.SetUpProblemIC_modes(p, *_modes(seed, (c["nx"], c["ny"], c["nz"]), _box(c), c["mhd"]))
    if c["kind"] == "forced":
        M.SetUpN97(p, F0=1, kf=2)
    state["sol"] = _sol_view(p, c["bits"])
    return state


# ---- one pass ------------------------------------------------------------------------------------
def run(state):
    c = state["case"]
    if c["kind"] == "ens":
        e = state["e"]
        e.step(c["steps"])
        return [e.get_sol(i) for i in range(len(e))]
    p = state["p"]
    if c["kind"] == "rhs":
        M.calcN(p, state["N"], state["sol"])
        return {"N": state["N"], "sol": state["sol"]}
    if c["kind"] == "step":
        M.stepforward(p, c["steps"])
        return {"sol": state["sol"]}
    M.TimeIntegrator(p, INF, c["steps"] - 1, CFL_Coef=CFL)
    if c["kind"] == "adv":
        return {"sol": state["sol"], "t": p.clock.t}
    d = M.Diagnostics(p)
    return {"sol": state["sol"], "t": p.clock.t,
            "diag": np.array([d[k] for k in ("E_kin", "E_mag", "H_kin", "H_mag", "H_cross")])}


def _modes_kept(n):
    lo, hi = _aliased(n)
    return lo + n - hi


def _work_one(shape, mhd, bits, rhs, steps):
    """Every right-hand side reads the kept modes of its input and writes those of its update once (a
    transform in three dimensions needs the whole field, so nothing smaller stays on the chip); the last
    state is written whole.  Operations: the transforms (5/2 N log2 N each, six inverse and nine forward
    for MHD, three and six for HD), the products and the update of each mode."""
    nx, ny, nz = shape
    nf, ntr = (6, 15) if mhd else (3, 9)
    n = float(nx * ny * nz)
    kept = _aliased(nx)[0] * _modes_kept(ny) * _modes_kept(nz)
    nc = (nx // 2 + 1) * ny * nz
    cx = bits // 4
    return {"bytes": cx * nf * (2.0 * kept * rhs + (nc if steps else 0)),
            "flops": rhs * (ntr * 2.5 * n * math.log2(n) + (27 if mhd else 6) * n + 100.0 * kept)}


def work(case):
    c = case
    stages = 4 if c["stepper"] == "RK4" else 5
    if c["kind"] == "ens":
        parts = [_work_one((n, n, n), True, c["bits"], stages * c["steps"], c["steps"]) for n in _sizes(c)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    shape = (c["nx"], c["ny"], c["nz"])
    if c["kind"] == "rhs":
        w = _work_one(shape, c["mhd"], c["bits"], 1, 0)
        nc = (c["nx"] // 2 + 1) * c["ny"] * c["nz"]
        return {"bytes": c["bits"] // 4 * (6 if c["mhd"] else 3) * 2.0 * nc, "flops": w["flops"]}
    return _work_one(shape, c["mhd"], c["bits"], stages * c["steps"], c["steps"])


# ---- the same in 64 bits, in plain torch -----------------------------------------------------------
def _aliased(n):
    """The band [lo, hi) of indices of an axis of n points that the 1/3 rule removes."""
    a = 1.0 / 3.0
    return math.floor((1.0 - a) / 2.0 * n), math.ceil((1.0 + a) / 2.0 * n)


class _Exact:
    """The right-hand side and steppers of ``runs`` runs of one grid on states [run, field, z, y, kx]."""

    def __init__(self, shape, box, mhd, nu, nnu, force=None):
        self.shape, self.box, self.mhd, self.nnu, self.force = shape, box, mhd, nnu, force
        self.k = _wavenumbers(shape, box, "cuda")
        self.k2 = self.k[0] ** 2 + self.k[1] ** 2 + self.k[2] ** 2
        self.inv = torch.where(self.k2 == 0, torch.zeros_like(self.k2), 1.0 / self.k2)
        self.nu = torch.as_tensor(nu, dtype=torch.float64, device="cuda").view(-1, 1, 1, 1)
        keep = [torch.ones(n, dtype=torch.float64, device="cuda") for n in (shape[0] // 2 + 1, shape[1], shape[2])]
        for v, n, half in zip(keep, shape, (True, False, False)):
            lo, hi = _aliased(n)
            v[lo:(None if half else hi)] = 0
        self.mask = keep[0][None, None, :] * keep[1][None, :, None] * keep[2][:, None, None]

    def hermitian(self, s):
        """The part of a masked state that a real field sees: the mask keeps index -n/3 of the y and z axes
        and not its mirror, so the kx = 0 plane is projected on its Hermitian part."""
        s = s.clone()
        p = s[..., 0]
        s[..., 0] = 0.5 * (p + torch.roll(p.flip(-1, -2), (1, 1), (-1, -2)).conj())
        return s

    def real(self, s):
        nx, ny, nz = self.shape
        return [torch.fft.irfftn(s[:, f], s=(nz, ny, nx), dim=(1, 2, 3)) for f in range(s.shape[1])]

    def rhs(self, s):
        """N of a masked state, and its real fields."""
        s = self.hermitian(s)
        v = self.real(s)
        k, N = self.k, torch.zeros_like(s)
        for i in range(3):
            for j in range(i, 3):
                T = v[3 + i] * v[3 + j] - v[i] * v[j] if self.mhd else -v[i] * v[j]
                T = torch.fft.rfftn(T, dim=(1, 2, 3)) * 1j
                N[:, j] += k[i] * T
                if i != j:
                    N[:, i] += k[j] * T
        p = (N[:, 0] * k[0] + N[:, 1] * k[1] + N[:, 2] * k[2]) * self.inv
        for i in range(3):
            N[:, i] -= k[i] * p
        if self.mhd:
            for i in range(3):
                for j in range(i + 1, 3):
                    m = torch.fft.rfftn(v[i] * v[3 + j] - v[3 + i] * v[j], dim=(1, 2, 3)) * 1j
                    N[:, 3 + i] += k[j] * m
                    N[:, 3 + j] -= k[i] * m
        damp = [self.k2 + (self.k2 ** self.nnu if self.nnu > 1 else 0), self.k2]  # hyperviscosity acts on u
        for f in range(s.shape[1]):
            N[:, f] -= damp[f // 3] * self.nu * s[:, f]
        if self.force is not None:
            N[:, :3] += self.force
        return N, v

    def largest(self, v):
        return torch.stack([x.abs().amax(dim=(1, 2, 3)) for x in v]).amax(0)

    def advance(self, s, stepper, steps, cfl=None, dt=None):
        """The state, the time and the real fields of the last stage's input after ``steps`` steps."""
        dl = min(L / n for L, n in zip(self.box, self.shape))
        nu = self.nu.view(-1)
        slow = cfl and cfl * dl ** (self.nnu if self.nnu > 1 else 2) / nu
        t = torch.zeros(s.shape[0], dtype=torch.float64, device="cuda")
        v = self.real(self.hermitian(s * self.mask))
        for _ in range(steps):
            h = torch.minimum(cfl * dl / self.largest(v), slow) if cfl else torch.full_like(t, dt)
            t = t + h
            h = h.view(-1, 1, 1, 1, 1)
            s = s * self.mask
            if stepper == "RK4":
                x, acc = s, 0
                for a, b in ((0.5, 1 / 6), (0.5, 1 / 3), (1.0, 1 / 3), (0.0, 1 / 6)):
                    del v
                    N, v = self.rhs(x)
                    acc = acc + b * N
                    x = (s + (a * h) * N) * self.mask if a else None
                s = s + h * acc
            else:
                S = 0
                for a, b in zip(_LSRK_A, _LSRK_B):
                    s = s * self.mask
                    del v
                    N, v = self.rhs(s)
                    S = a * S + h * N
                    s = s + b * S
        return s, t, v


# Carpenter and Kennedy's five-stage fourth-order low-storage scheme
_LSRK_A = (0.0, -567301805773 / 1357537059087, -2404267990393 / 2016746695238, -3550918686646 / 2091501179385,
           -1275806237668 / 842570457699)
_LSRK_B = (1432997174477 / 9575080441755, 5161836677717 / 13612068292357, 1720146321549 / 2090206949498,
           3134564353537 / 4481467310338, 2277821191437 / 14882151754819)


def _dense(idx, vals, shape, bits):
    """Sparse entries as a state in 64 bits, its values rounded as the framework takes them."""
    nf = vals.shape[1]
    s = torch.zeros(nf, shape[2], shape[1], shape[0] // 2 + 1, dtype=torch.complex128, device="cuda")
    v = torch.from_numpy(vals).to("cuda")
    v = v.to(torch.complex64).to(torch.complex128) if bits == 32 else v
    i = torch.from_numpy(idx.astype(np.int64)).to("cuda")
    s[:, i[:, 2], i[:, 1], i[:, 0]] = v.T
    return s


def exact(case, seed):
    c = case
    with torch.no_grad():
        if c["kind"] == "ens":
            params, sizes = _run_params(c, seed), _sizes(c)
            out = [None] * len(sizes)
            for n in sorted(set(sizes)):
                mine = [i for i, v in enumerate(sizes) if v == n]
                s = torch.stack([_dense(*_modes(seed * 1000 + i, (n, n, n), (2 * math.pi,) * 3, True, params[i][1]),
                                        (n, n, n), c["bits"]) for i in mine])
                e = _Exact((n, n, n), (2 * math.pi,) * 3, True, [params[i][0] for i in mine], 0)
                s = e.advance(s, c["stepper"], c["steps"], cfl=CFL)[0]
                for j, i in enumerate(mine):
                    out[i] = s[j].cpu().numpy()
            return out
        shape, box = (c["nx"], c["ny"], c["nz"]), _box(c)
        if c["kind"] == "rhs":
            e = _Exact(shape, box, c["mhd"], [c["nu"]], c["nnu"])
            s = _dense_state(c, seed).to(torch.complex128) * e.mask
            return {"N": e.rhs(s[None])[0][0], "sol": s}
        force = None
        if c["kind"] == "forced":
            x, y, z = (torch.as_tensor(-L / 2 + np.arange(n) * (L / n), device="cuda") for L, n in zip(box, shape))
            x, y, z = 2 * x[None, None, :], 2 * y[None, :, None], 2 * z[:, None, None]
            f = torch.stack([x.sin() * y.cos() * z.cos(), -x.cos() * y.sin() * z.cos(), 0 * (x + y + z)])
            force = torch.fft.rfftn(f, dim=(1, 2, 3))
        e = _Exact(shape, box, c["mhd"], [c["nu"]], c["nnu"], force)
        s = _dense(*_modes(seed, shape, box, c["mhd"]), shape, c["bits"])[None]
        if c["kind"] == "step":
            dt = float(_np_type(c)(_fixed_dt(c)))
            return {"sol": e.advance(s, c["stepper"], c["steps"], dt=dt)[0][0]}
        s, t, v = e.advance(s, c["stepper"], c["steps"], cfl=CFL)
        got = {"sol": s[0], "t": float(t[0])}
        if c["kind"] == "forced":
            dV = float(np.prod([L / n for L, n in zip(box, shape)]))
            u, b = v[:3], v[3:]
            w, a = _curl(e, u), _curl(e, b, e.inv)
            dot = lambda p, q: float(sum((x * y).sum() for x, y in zip(p, q))) * dV  # noqa: E731
            got["diag"] = np.array([dot(u, u), dot(b, b), dot(w, u), dot(a, b), dot(u, b)])
        return got


def _curl(e, v, scale=1.0):
    """curl of real fields; times ``scale`` in spectral space (1 / k^2: the vector potential)."""
    h = [torch.fft.rfftn(x, dim=(1, 2, 3)) * scale for x in v]
    k = e.k
    c = [1j * (k[1] * h[2] - k[2] * h[1]), 1j * (k[2] * h[0] - k[0] * h[2]), 1j * (k[0] * h[1] - k[1] * h[0])]
    return e.real(torch.stack(c, 1))
