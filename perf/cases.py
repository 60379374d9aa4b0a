"""Timed workloads of the library, one pass through its public entry points each.

``listed()`` names the workloads, ``draw(rng)`` gives another one of the same
ranges, ``prepare(case, seed)`` builds what a program holds before the call
(model and state on the GPU), ``run(state)`` makes one pass and returns every
output, ``work(case)`` counts the bytes and operations the pass cannot do
without, and ``exact(case, seed)`` evaluates the same pass in FP64 with plain
torch.

A case names a kind of model (``barotropic``, ``baroclinic``, ``ensemble``,
``swm``, ``nonlinear_swm``, ``masked``), its grid, its options and the call.
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

import somax_amd
from somax_amd.elliptic import MaskedHelmholtz, octagon_node_mask

BASIN = 5.12e6  # double-gyre basin (m)
F0, BETA = 9.375e-5, 1.754e-11
DEPTHS = {1: (4000.0,), 2: (400.0, 3600.0), 3: (400.0, 1100.0, 2600.0)}
GRAVITIES = {1: (9.81,), 2: (9.81, 0.025), 3: (9.81, 0.025, 0.0125)}
# members of the ensemble: the 96/96/48/16 mix of 64^2..512^2 grids, an eighth of it
ENSEMBLE = ((64, 12), (128, 12), (256, 6), (512, 2))
TSIT5 = (
    (0.161,),
    (-0.008480655492356989, 0.335480655492357),
    (2.897153057105493, -6.359448489975075, 4.3622954328695815),
    (5.325864828439257, -11.748883564062828, 7.4955393428898365, -0.09249506636175525),
    (5.86145544294642, -12.92096931784711, 8.159367898576159, -0.071584973281401, -0.028269050394068383),
    (0.09646076681806523, 0.01, 0.4798896504144996, 1.379008574103742, -3.290069515436081, 2.324710524099774),
)


def _qg(name, op, nx, ny, nl, precision, advection="arakawa", mass=False, solver="ssprk3", steps=1, kind="baroclinic"):
    return {"name": name, "kind": kind, "op": op, "nx": nx, "ny": ny, "nl": nl, "precision": precision,
            "advection": advection, "mass": mass, "solver": solver, "steps": steps, "dt": 1200.0}


def _swm(name, op, nx, ny, nl, bc, flux="average", solver="ssprk3", steps=1, kind="swm"):
    return {"name": name, "kind": kind, "op": op, "nx": nx, "ny": ny, "nl": nl, "bc": bc, "flux": flux,
            "solver": solver, "steps": steps}


def listed():
    return [
        # the reference's CPU configuration: one step of the 64^2 barotropic gyre in FP64
        _qg("barotropic_64_fp64_step", "step", 64, 64, 1, "fp64", kind="barotropic"),
        # the barotropic gyre as a new user runs it: defaults (FP32), integrate with its default solver
        _qg("barotropic_64_fp32_integrate", "integrate", 64, 64, 1, "fp32", solver="tsit5", steps=4, kind="barotropic"),
        # the multilayer double gyre at its default size and solver
        _qg("gyre_3x128_fp32_integrate", "integrate", 128, 128, 3, "fp32", solver="tsit5", steps=2),
        # spin-up runs at 256^2 with WENO-Z fluxes and the mass constraint
        _qg("gyre_3x256_weno_mass_mixed_step", "step", 256, 256, 3, "mixed", "weno", True),
        # a larger run with the default precision and advection
        _qg("gyre_3x512_fp32_step", "step", 512, 512, 3, "fp32"),
        # the benchmark workload: eddy-resolving, mixed-precision inversion
        _qg("gyre_3x1024_weno_mass_mixed_step", "step", 1024, 1024, 3, "mixed", "weno", True),
        # one right-hand side for an outside integrator, on a grid of odd, unequal sides
        _qg("gyre_2x301x216_fp32_rhs", "rhs", 301, 216, 2, "fp32"),
        # diagnostics of a run (inversion, velocities, energies) with the six-product transforms
        _qg("gyre_3x512_bf16x6_diagnose", "diagnose", 512, 512, 3, "bf16x6"),
        # an uneven ensemble, one step of all members
        {"name": "ensemble_32_mixed_step", "kind": "ensemble", "op": "step", "counts": 1, "precision": "mixed",
         "advection": "weno", "mass": True, "solver": "ssprk3", "steps": 1, "dt": 1200.0},
        # the shallow-water jet in a channel
        _swm("swm_2x512_channel_een_step", "step", 512, 512, 2, "channel", "energy_enstrophy"),
        # a small shallow-water run with the default boundary condition and solver
        _swm("swm_3x64_periodic_integrate", "integrate", 64, 64, 3, "periodic", solver="tsit5", steps=4),
        # Helmholtz solve on an octagonal basin
        {"name": "octagon_3x128_mixed_solve", "kind": "masked", "op": "solve", "nx": 128, "ny": 128, "nl": 3,
         "precision": "mixed"},
    ]


def _size(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(max(n + rng.choice((0, 0, 1)), lo), hi)


def draw(rng):
    kind = rng.choice(("barotropic", "baroclinic", "baroclinic", "baroclinic", "swm", "nonlinear_swm", "masked",
                       "ensemble"))
    if kind == "ensemble":
        return {"kind": kind, "op": "step", "counts": 1, "precision": rng.choice(("mixed", "fp32", "bf16x6")),
                "advection": rng.choice(("weno", "arakawa")), "mass": rng.choice((True, False)), "solver": "ssprk3",
                "steps": 1, "dt": float(rng.choice((600.0, 900.0, 1200.0)))}
    if kind == "masked":
        n = _size(rng, 32, 128)
        return {"kind": kind, "op": "solve", "nx": n, "ny": min(128, max(32, n + rng.randint(-8, 8))),
                "nl": rng.randint(1, 3), "precision": rng.choice(("mixed", "fp32", "bf16x6"))}
    if kind in ("swm", "nonlinear_swm"):
        n = _size(rng, 32, 512)
        nl = rng.randint(1, 3) if kind == "swm" else 1
        bc = rng.choice(("periodic", "wall", "channel")) if kind == "swm" else rng.choice(("periodic", "wall"))
        c = _swm("", rng.choice(("step", "step", "integrate", "rhs")), n, _size(rng, max(32, n // 2), min(512, 2 * n)), nl,
                 bc, rng.choice(("average", "energy_enstrophy")) if kind == "swm" else "average",
                 rng.choice(("ssprk3", "tsit5")), rng.randint(1, 3), kind)
    elif kind == "barotropic":
        n = _size(rng, 32, 256)
        c = _qg("", rng.choice(("step", "integrate", "rhs", "diagnose")), n, _size(rng, max(32, n // 2), 2 * n), 1,
                rng.choice(("fp32", "fp64", "mixed")), rng.choice(("arakawa", "weno")), False,
                rng.choice(("ssprk3", "tsit5")), rng.randint(1, 3), kind)
    else:
        n = _size(rng, 48, 768)
        c = _qg("", rng.choice(("step", "step", "rhs", "diagnose")), n, _size(rng, max(48, n // 2), min(768, 2 * n)),
                rng.randint(1, 3), rng.choice(("fp32", "fp32", "mixed", "mixed", "bf16x6")),
                rng.choice(("arakawa", "weno")), rng.choice((True, False)), "ssprk3", 1, kind)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# models and inputs
# ---------------------------------------------------------------------------
def _qg_args(case, nx=None, nl=None, tau0=0.08):
    """``create`` arguments of a QG case (square cells on the basin)."""
    if nx is None:
        nx, ny, nl = case["nx"], case["ny"], case["nl"]
    else:
        ny = nx
    Ly = BASIN * ny / nx
    kw = dict(nx=nx, ny=ny, Lx=BASIN, Ly=Ly, f0=F0, beta=BETA, bottom_drag=3.6e-8,
              biharmonic_viscosity=2e11 * (128.0 / nx) ** 4, lateral_viscosity=15.0,
              wind_amplitude=tau0 * 2.0 * math.pi / (1000.0 * Ly))
    if case["kind"] == "barotropic":
        kw["wind_amplitude"] /= 4000.0
    else:
        kw.update(n_layers=nl, H=DEPTHS[nl], g_prime=GRAVITIES[nl])
    return kw


def _qg_model(case, kw):
    opts = dict(advection=case["advection"], precision=case["precision"])
    if case["kind"] == "barotropic":
        return somax_amd.BarotropicQG.create(**kw, **opts)
    return somax_amd.BaroclinicQG.create(**kw, **opts, mass_correction=case["mass"])


def _dst_sum(c, axis):
    """sum_k c_k sin(pi j k / (n + 1)) along an axis, by an FFT of the odd extension."""
    c = np.moveaxis(c, axis, -1)
    n = c.shape[-1]
    z = np.zeros(c.shape[:-1] + (2 * n + 2,))
    z[..., 1:n + 1] = c
    z[..., n + 2:] = -c[..., ::-1]
    return np.moveaxis(-0.5 * np.fft.rfft(z, axis=-1).imag[..., 1:n + 1], -1, axis)


def _random_psi(kw, nl, seed, zero_mean):
    """A seeded k^-3 streamfunction of 0.05 m/s rms speed per layer, zero on the ghost ring."""
    nx, ny, dx, dy = kw["nx"], kw["ny"], kw["Lx"] / kw["nx"], kw["Ly"] / kw["ny"]
    rng = np.random.default_rng(seed)
    k = np.hypot((np.arange(1, ny + 1) / ((ny + 1) * dy))[:, None], (np.arange(1, nx + 1) / ((nx + 1) * dx))[None])
    psi = np.zeros((nl, ny + 2, nx + 2))
    psi[:, 1:-1, 1:-1] = _dst_sum(_dst_sum(rng.standard_normal((nl, ny, nx)) * (k / k.min()) ** -3.0, -1), -2)
    if zero_mean:
        g = np.sin(np.pi * np.arange(ny + 2) / (ny + 1))[:, None] * np.sin(np.pi * np.arange(nx + 2) / (nx + 1))
        psi -= psi.mean(axis=(1, 2), keepdims=True) / g.mean() * g
    speed2 = ((np.diff(psi, axis=1)[:, 1:, 1:-1] / dy) ** 2 + (np.diff(psi, axis=2)[:, 1:-1, 1:] / dx) ** 2).mean(axis=(1, 2))
    return psi * (0.05 / np.sqrt(speed2))[:, None, None]


def _random_q(case, kw, nl, seed):
    """The PV of a random streamfunction, float64."""
    psi = _random_psi(kw, nl, seed, case["mass"])
    _, _, lam, l2m, m2l = _modes(case["kind"], nl)
    q = np.zeros_like(psi)
    c = psi[:, 1:-1, 1:-1]
    q[:, 1:-1, 1:-1] = ((psi[:, 1:-1, 2:] - 2 * c + psi[:, 1:-1, :-2]) / (kw["Lx"] / kw["nx"]) ** 2
                        + (psi[:, 2:, 1:-1] - 2 * c + psi[:, :-2, 1:-1]) / (kw["Ly"] / kw["ny"]) ** 2
                        - np.einsum("lk,kyx->lyx", m2l @ np.diag(lam) @ l2m, c))
    return q


def _members(case, seed):
    """(create arguments, layers, seed) of every ensemble member."""
    rng = np.random.default_rng(seed)
    out = []
    for n, count in ENSEMBLE:
        for _ in range(count * case["counts"]):
            nl = 1 + len(out) % 3
            out.append((_qg_args(case, n, nl, float(rng.uniform(0.04, 0.12))), nl, seed * 1009 + len(out)))
    return out


def _swm_args(case):
    L = 4000.0 * case["nx"]
    kw = dict(nx=case["nx"], ny=case["ny"], Lx=L, Ly=4000.0 * case["ny"], f0=1e-4, beta=BETA, bottom_drag=1e-7,
              lateral_viscosity=50.0, bc=case["bc"])
    if case["kind"] == "nonlinear_swm":
        return dict(kw, H0=500.0, wind_amplitude=1e-7)
    nl = case["nl"]
    return dict(kw, n_layers=nl, H=DEPTHS[nl], g_prime=GRAVITIES[nl], wind_amplitude=1e-4,
                vorticity_flux=case["flux"])


def _swm_dt(case):
    return 0.3 * 4000.0 / math.sqrt(9.81 * (500.0 if case["kind"] == "nonlinear_swm" else 4000.0))


def _swm_fields(case, seed):
    """Thickness, velocities: smooth waves of metres and tenths of m/s plus small noise, float32."""
    rng = np.random.default_rng(seed)
    nl, ny, nx = case["nl"], case["ny"], case["nx"]
    H = (500.0,) if case["kind"] == "nonlinear_swm" else DEPTHS[nl]
    y, x = np.arange(ny + 2) / ny, np.arange(nx + 2) / nx
    out = []
    for scale, noise in ((2.0, 0.2), (0.3, 0.02), (0.3, 0.02)):
        f = np.zeros((nl, ny + 2, nx + 2))
        for ky in range(1, 5):
            for kx in range(1, 5):
                a, p, r = rng.standard_normal(nl), rng.uniform(0, 2 * np.pi), rng.uniform(0, 2 * np.pi)
                f += (a / (ky * ky + kx * kx))[:, None, None] * (
                    np.sin(2 * np.pi * ky * y + p)[:, None] * np.sin(2 * np.pi * kx * x + r))
        out.append(scale * f + noise * (rng.random(f.shape) - 0.5))
    out[0] += np.asarray(H)[:, None, None]
    return [a.astype(np.float32) for a in out]


def _masked_args(case):
    nl = case["nl"]
    A = _coupling(DEPTHS[nl], GRAVITIES[nl])
    A[0, 0] -= 1.0 / (DEPTHS[nl][0] * GRAVITIES[nl][0])  # rigid lid
    d = BASIN / (case["nx"] - 1)
    return octagon_node_mask(case["nx"], case["ny"]), d, F0**2 * np.maximum(np.sort(np.linalg.eigvals(A).real), 0.0)


def _cuda(a, dtype=torch.float32):
    return torch.as_tensor(np.ascontiguousarray(a)).to(dtype).to("cuda")


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "ensemble":
        members = _members(case, seed)
        models = [_qg_model(case, kw) for kw, _, _ in members]
        st["ens"] = somax_amd.QGEnsemble(models)
        st["q0"] = st["ens"].pack([_random_q(case, kw, nl, s).astype(np.float32) for kw, nl, s in members])
        st["q"] = st["q0"].clone()
    elif kind == "masked":
        mask, d, lam = _masked_args(case)
        st["solver"] = MaskedHelmholtz(mask, d, d, lam, precision=case["precision"])
        st["rhs"] = _cuda(_masked_rhs(case, seed))
    elif kind in ("swm", "nonlinear_swm"):
        h, u, v = (_cuda(a) for a in _swm_fields(case, seed))
        if kind == "swm":
            st["model"] = somax_amd.MultilayerShallowWater2D.create(**_swm_args(case))
            st["y"] = somax_amd.MultilayerSW2DState(h=h, u=u, v=v)
        else:
            st["model"] = somax_amd.NonlinearShallowWater2D.create(**_swm_args(case))
            st["y"] = somax_amd.NonlinearSW2DState(h=h[0].contiguous(), u=u[0].contiguous(), v=v[0].contiguous())
        st["dt"] = _swm_dt(case)
    else:
        kw = _qg_args(case)
        st["model"] = _qg_model(case, kw)
        q = _cuda(_random_q(case, kw, case["nl"], seed).astype(np.float32),
                  torch.float64 if case["precision"] == "fp64" else torch.float32)
        st["y"] = (somax_amd.BarotropicQGState(q=q[0].contiguous()) if kind == "barotropic"
                   else somax_amd.BaroclinicQGState(q=q))
        st["dt"] = case["dt"]
    return st


def _masked_rhs(case, seed):
    return (np.random.default_rng(seed).standard_normal((case["nl"], case["ny"], case["nx"])) * 1e-10).astype(np.float32)


def run(state):
    case = state["case"]
    op = case["op"]
    if case["kind"] == "ensemble":
        state["q"].copy_(state["q0"])  # the members' start state, stepped in place
        state["ens"].step(state["q"], case["dt"], case["steps"])
        return state["ens"].unpack(state["q"])
    if case["kind"] == "masked":
        return state["solver"].solve(state["rhs"])
    model, y, dt = state["model"], state["y"], state["dt"]
    if op == "step":
        out = model.step(y, dt, case["steps"], solver=case["solver"])
    elif op == "integrate":
        out = model.integrate(y, 0.0, case["steps"] * dt, dt, solver=case["solver"]).ys
    elif op == "rhs":
        out = model.build_terms()(0.0, y, None)
    else:
        d = model.diagnose(y)
        return [d.psi, d.u, d.v, d.relative_vorticity, d.kinetic_energy, d.enstrophy]
    return [out.q] if hasattr(out, "q") else [out.h, out.u, out.v]


# ---------------------------------------------------------------------------
# necessary work
# ---------------------------------------------------------------------------
def _evaluations(case):
    if case["op"] in ("rhs", "diagnose"):
        return 1
    return case["steps"] * (3 if case["solver"] == "ssprk3" else 6)


def _qg_work(case, nx, ny, nl):
    """Bytes: the state read once and every output written once.  Operations
    per evaluation: two sine transforms there and back by a fast transform
    (2.5 M log2 M for the odd extension of M points), the projections and the
    stencils."""
    word = 8 if case["precision"] == "fp64" else 4
    cells = (nx + 2) * (ny + 2) * nl
    arrays = 5 if case["op"] == "diagnose" else 2
    per_cell = 2 * 2.5 * (math.log2(2 * nx + 6) + math.log2(2 * ny + 6)) * 2 + 4 * nl
    if case["op"] != "diagnose":
        per_cell += 160 if case["advection"] == "weno" else 90
    return word * cells * arrays, per_cell * cells * _evaluations(case)


def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        parts = [_qg_work(case, n, n, 1 + i % 3)
                 for i, n in enumerate(n for n, count in ENSEMBLE for _ in range(count * case["counts"]))]
        return {"bytes": float(sum(p[0] for p in parts)), "flops": float(sum(p[1] for p in parts))}
    if kind == "masked":
        mask, _, lam = _masked_args(case)
        m = somax_amd.irregular_boundary(mask)[0].size
        cells = case["nx"] * case["ny"] * case["nl"]
        lg = math.log2(2 * case["nx"] + 2) + math.log2(2 * case["ny"] + 2)
        return {"bytes": float(8 * cells + 8 * m * m * case["nl"]),
                "flops": float(2 * 10.0 * lg * cells + 2.0 * m * m * case["nl"])}
    if kind in ("swm", "nonlinear_swm"):
        cells = (case["nx"] + 2) * (case["ny"] + 2) * case["nl"]
        return {"bytes": float(4 * 6 * cells),
                "flops": float((140 if case["flux"] == "energy_enstrophy" else 110) * cells * _evaluations(case))}
    b, f = _qg_work(case, case["nx"], case["ny"], case["nl"])
    return {"bytes": float(b), "flops": float(f)}


# ---------------------------------------------------------------------------
# the same passes in FP64 with plain torch
# ---------------------------------------------------------------------------
def _coupling(H, gp):
    nl = len(H)
    A = np.zeros((nl, nl))
    for k in range(nl):
        A[k, k] = 1.0 / (H[k] * gp[k])
        if k:
            A[k, k - 1] = -1.0 / (H[k] * gp[k])
        if k + 1 < nl:
            A[k, k] += 1.0 / (H[k] * gp[k + 1])
            A[k, k + 1] = -1.0 / (H[k] * gp[k + 1])
    return A


@functools.lru_cache(maxsize=None)
def _modes(kind, nl):
    """(H, g', Helmholtz parameter per mode, layer->mode, mode->layer) in FP64."""
    if kind == "barotropic":
        return None, None, np.zeros(1), np.eye(1), np.eye(1)
    w, R = np.linalg.eig(_coupling(DEPTHS[nl], GRAVITIES[nl]))
    order = np.argsort(w.real)
    R = R.real[:, order]
    return DEPTHS[nl], GRAVITIES[nl], F0**2 * w.real[order], np.linalg.inv(R), R


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _f64(a):
    return torch.as_tensor(a, dtype=torch.float64, device=_device())


def _sine(n):
    # integer angles reduced modulo one period, so large n keeps full accuracy
    k = torch.arange(1, n + 1, dtype=torch.int64, device=_device())
    a = torch.remainder(k[:, None] * k[None, :], 2 * (n + 1)).double()
    return math.sqrt(2.0 / (n + 1)) * torch.sin(math.pi / (n + 1) * a)


def _eig(n, d):
    k = torch.arange(1, n + 1, dtype=torch.float64, device=_device())
    return -4.0 * torch.sin(0.5 * math.pi * k / (n + 1)) ** 2 / (d * d)


def _lap(f, dx, dy):
    out = torch.zeros_like(f)
    c = f[..., 1:-1, 1:-1]
    out[..., 1:-1, 1:-1] = ((f[..., 1:-1, 2:] - 2 * c + f[..., 1:-1, :-2]) / dx**2
                            + (f[..., 2:, 1:-1] - 2 * c + f[..., :-2, 1:-1]) / dy**2)
    return out


def _inside(q):
    out = torch.zeros_like(q)
    out[..., 1:-1, 1:-1] = q[..., 1:-1, 1:-1]
    return out


def _weno_faces(q, vel):
    """Upwind WENO-Z values at the n-1 inner faces along the last axis."""
    n = q.shape[-1]
    p = torch.cat([q[..., :1], q[..., :1], q, q[..., -1:], q[..., -1:]], dim=-1)
    f = torch.arange(1, n, device=q.device)

    def five(a, b, c, d, e):
        b0 = 13 / 12 * (a - 2 * b + c) ** 2 + 0.25 * (a - 4 * b + 3 * c) ** 2
        b1 = 13 / 12 * (b - 2 * c + d) ** 2 + 0.25 * (b - d) ** 2
        b2 = 13 / 12 * (c - 2 * d + e) ** 2 + 0.25 * (3 * c - 4 * d + e) ** 2
        tau = (b0 - b2).abs()
        w = [g * (1 + tau / (b_ + 1e-20)) for g, b_ in ((0.1, b0), (0.6, b1), (0.3, b2))]
        v = ((2 * a - 7 * b + 11 * c) / 6, (-b + 5 * c + 2 * d) / 6, (2 * c + 5 * d - e) / 6)
        return sum(x * y for x, y in zip(w, v)) / sum(w)

    def three(b, c, d):
        b0, b1 = (c - b) ** 2, (d - c) ** 2
        tau = (b0 - b1).abs()
        w = [g * (1 + tau / (b_ + 1e-20)) for g, b_ in ((1 / 3, b0), (2 / 3, b1))]
        return (w[0] * (3 * c - b) / 2 + w[1] * (c + d) / 2) / (w[0] + w[1])

    def side(cells, up):
        s = [p[..., 2 + o:1 + n + o] for o in cells]
        return torch.where((up >= 3) & (up <= n - 2), five(*s),
                           torch.where((up >= 2) & (up <= n - 1), three(*s[1:4]), s[2]))

    return torch.where(vel > 0, side((-2, -1, 0, 1, 2), f), side((3, 2, 1, 0, -1), f + 1))


class _QGExact:
    def __init__(self, case, kw, nl):
        self.case, self.kw, self.nl = case, kw, nl
        self.nx, self.ny = kw["nx"], kw["ny"]
        self.dx, self.dy = kw["Lx"] / self.nx, kw["Ly"] / self.ny
        H, _, lam, l2m, m2l = _modes(case["kind"], nl)
        self.Sx, self.Sy = _sine(self.nx + 2), _sine(self.ny + 2)
        self.lam, self.l2m, self.m2l = _f64(lam), _f64(l2m), _f64(m2l)
        self.den = (_eig(self.ny + 2, self.dy)[:, None] + _eig(self.nx + 2, self.dx)[None])[None] - self.lam[:, None, None]
        y = _f64(np.arange(self.ny + 2) * self.dy)
        self.b = (BETA * (y - kw["Ly"] / 2))[:, None]
        scale = np.zeros(nl)
        scale[0] = 1.0 if H is None else 1.0 / H[0]
        self.wind = (kw["wind_amplitude"] * _f64(scale)[:, None, None] * -torch.sin(2 * math.pi * y / kw["Ly"])[None, :, None])
        self.mass = case["mass"]
        if self.mass:
            self.h = 1 + self._solve(self.lam[:, None, None] * torch.ones_like(self.den))

    def _solve(self, f):
        return self.Sy @ ((self.Sy @ f @ self.Sx) / self.den) @ self.Sx

    def invert(self, q):
        pm = self._solve(torch.einsum("mk,kyx->myx", self.l2m, q))
        wall = torch.zeros(self.nl, dtype=torch.float64, device=q.device)
        if self.mass:
            alpha = -pm.mean(dim=(1, 2)) / self.h.mean(dim=(1, 2))
            pm = pm + alpha[:, None, None] * self.h
            wall = self.m2l @ alpha
        psi = torch.einsum("lm,myx->lyx", self.m2l, pm)
        return (psi if self.mass or self.case["kind"] == "barotropic" else _inside(psi)), wall

    def rhs(self, q):
        dx, dy, kw = self.dx, self.dy, self.kw
        q = _inside(q)
        psi, wall = self.invert(q)
        t = q + self.b
        dq = torch.zeros_like(q)
        if self.case["advection"] == "weno":
            c = 0.25 * (psi[:, :-1, :-1] + psi[:, :-1, 1:] + psi[:, 1:, :-1] + psi[:, 1:, 1:])
            c[:, (0, -1), :] = wall[:, None, None]
            c[:, :, (0, -1)] = wall[:, None, None]
            u = -(c[:, 1:, 1:-1] - c[:, :-1, 1:-1]) / dy
            v = (c[:, 1:-1, 1:] - c[:, 1:-1, :-1]) / dx
            ti = t[:, 1:-1, 1:-1]
            fx = torch.nn.functional.pad(u * _weno_faces(ti, u), (1, 1))
            fy = torch.nn.functional.pad(v * _weno_faces(ti.transpose(1, 2), v.transpose(1, 2)).transpose(1, 2), (0, 0, 1, 1))
            dq[:, 1:-1, 1:-1] = -(fx[..., 1:] - fx[..., :-1]) / dx - (fy[:, 1:] - fy[:, :-1]) / dy
        else:
            def s(a, j, i):
                return a[:, 1 + j:self.ny + 1 + j, 1 + i:self.nx + 1 + i]

            E, W, N, S = (0, 1), (0, -1), (1, 0), (-1, 0)
            NE, NW, SE, SW = (1, 1), (1, -1), (-1, 1), (-1, -1)
            jpp = (s(psi, *E) - s(psi, *W)) * (s(t, *N) - s(t, *S)) - (s(psi, *N) - s(psi, *S)) * (s(t, *E) - s(t, *W))
            jpx = (s(psi, *E) * (s(t, *NE) - s(t, *SE)) - s(psi, *W) * (s(t, *NW) - s(t, *SW))
                   - s(psi, *N) * (s(t, *NE) - s(t, *NW)) + s(psi, *S) * (s(t, *SE) - s(t, *SW)))
            jxp = (s(t, *N) * (s(psi, *NE) - s(psi, *NW)) - s(t, *S) * (s(psi, *SE) - s(psi, *SW))
                   - s(t, *E) * (s(psi, *NE) - s(psi, *SE)) + s(t, *W) * (s(psi, *NW) - s(psi, *SW)))
            dq[:, 1:-1, 1:-1] = -(jpp + jpx + jxp) / (12 * dx * dy)
        lq = _lap(q, dx, dy)
        dq = dq + self.wind + kw["lateral_viscosity"] * lq - kw["biharmonic_viscosity"] * _lap(lq, dx, dy)
        dq[-1] -= kw["bottom_drag"] * _lap(psi[-1], dx, dy)
        return dq

    def diagnose(self, q):
        psi, _ = self.invert(q)
        dx, dy = self.dx, self.dy
        u, v = torch.zeros_like(psi), torch.zeros_like(psi)
        u[:, :-1] = -(psi[:, 1:] - psi[:, :-1]) / dy
        v[:, :, :-1] = (psi[:, :, 1:] - psi[:, :, :-1]) / dx
        uT, vT = 0.5 * (u[:, 1:-1, 1:-1] + u[:, :-2, 1:-1]), 0.5 * (v[:, 1:-1, 1:-1] + v[:, 1:-1, :-2])
        ke = 0.5 * (uT**2 + vT**2).sum(dim=(1, 2)) * dx * dy
        ens = 0.5 * (q[:, 1:-1, 1:-1] ** 2).sum(dim=(1, 2)) * dx * dy
        return psi, u, v, _lap(psi, dx, dy), ke, ens


def _advance(rhs, y, dt, steps, solver):
    """``steps`` steps of a tuple of fields."""
    for _ in range(steps):
        if solver == "tsit5":
            k = []
            for i in range(6):
                a = TSIT5[i - 1] if i else ()
                k.append(rhs(tuple(f + dt * sum((w * kj[n] for w, kj in zip(a, k)), 0.0) for n, f in enumerate(y))))
            y = tuple(f + dt * sum(w * kj[n] for w, kj in zip(TSIT5[5], k)) for n, f in enumerate(y))
        else:
            y1 = tuple(f + dt * d for f, d in zip(y, rhs(y)))
            y2 = tuple(0.75 * f + 0.25 * (g + dt * d) for f, g, d in zip(y, y1, rhs(y1)))
            y = tuple(f / 3 + 2 / 3 * (g + dt * d) for f, g, d in zip(y, y2, rhs(y2)))
    return y


class _SWMExact:
    def __init__(self, case):
        self.kw = kw = _swm_args(case)
        self.dx, self.dy, self.bc = kw["Lx"] / kw["nx"], kw["Ly"] / kw["ny"], case["bc"]
        self.een = case["flux"] == "energy_enstrophy"
        single = case["kind"] == "nonlinear_swm"
        H, gp = ((kw["H0"],), (9.81,)) if single else (kw["H"], kw["g_prime"])
        self.gp = _f64(gp)[:, None, None]
        y = _f64(np.arange(kw["ny"] + 2) * self.dy)
        f = (kw["f0"] + kw["beta"] * (y - kw["Ly"] / 2))[:, None]
        self.fX = 0.5 * (f[:-1] + f[1:])
        self.wind = kw["wind_amplitude"] / (1.0 if single else H[0]) * -torch.cos(2 * math.pi * y / kw["Ly"])[:, None]

    def boundary(self, y):
        h, u, v = (a.clone() for a in y)
        for name, a in (("h", h), ("u", u), ("v", v)):
            if self.bc == "periodic":
                a[:, 0], a[:, -1] = a[:, -2].clone(), a[:, 1].clone()
            elif name == "v":
                a[:, 0] = a[:, -2] = a[:, -1] = 0.0
            else:
                a[:, 0], a[:, -1] = a[:, 1].clone(), a[:, -2].clone()
            if self.bc != "wall":
                a[:, :, 0], a[:, :, -1] = a[:, :, -2].clone(), a[:, :, 1].clone()
            elif name == "u":
                a[:, :, 0] = a[:, :, -2] = a[:, :, -1] = 0.0
            else:
                a[:, :, 0], a[:, :, -1] = a[:, :, 1].clone(), a[:, :, -2].clone()
        return h, u, v

    def rhs(self, y):
        h, u, v = self.boundary(y)
        dx, dy, kw = self.dx, self.dy, self.kw
        F, G, uh, vh = (torch.zeros_like(h) for _ in range(4))
        hw, he, hs, hn = h[:, :, :-1], h[:, :, 1:], h[:, :-1], h[:, 1:]
        F[:, :, :-1] = u[:, :, :-1] * torch.where(u[:, :, :-1] > 0, hw, he)
        G[:, :-1] = v[:, :-1] * torch.where(v[:, :-1] > 0, hs, hn)
        uh[:, :, :-1] = 0.5 * (hw + he) * u[:, :, :-1]
        vh[:, :-1] = 0.5 * (hs + hn) * v[:, :-1]
        dh, du, dv = (torch.zeros_like(h) for _ in range(3))
        dh[:, 1:-1, 1:-1] = (-(F[:, 1:-1, 1:-1] - F[:, 1:-1, :-2]) / dx - (G[:, 1:-1, 1:-1] - G[:, :-2, 1:-1]) / dy)
        q = torch.zeros_like(h)
        hX = 0.25 * (h[:, :-1, :-1] + h[:, :-1, 1:] + h[:, 1:, :-1] + h[:, 1:, 1:])
        q[:, :-1, :-1] = ((v[:, :-1, 1:] - v[:, :-1, :-1]) / dx - (u[:, 1:, :-1] - u[:, :-1, :-1]) / dy + self.fX) / hX
        P = torch.cumsum(self.gp * h, dim=0)
        P[:, 1:, 1:] += 0.25 * (u[:, 1:, 1:] ** 2 + u[:, 1:, :-1] ** 2 + v[:, 1:, 1:] ** 2 + v[:, :-1, 1:] ** 2)

        def s(a, j, i):
            return a[:, 1 + j:a.shape[1] - 1 + j, 1 + i:a.shape[2] - 1 + i]

        if self.een:
            if self.bc != "wall":
                q[:, :, -1] = q[:, :, 1]
            if self.bc == "periodic":
                q[:, -1] = q[:, 1]
            tne = (s(q, 0, -1) + s(q, 0, 0) + s(q, -1, 0)) / 12
            tse = (s(q, 0, 0) + s(q, -1, 0) + s(q, -1, -1)) / 12
            tnw = (s(q, -1, -1) + s(q, 0, -1) + s(q, 0, 0)) / 12
            fu = (tne * s(vh, 0, 0) + tse * s(vh, -1, 0) + (s(q, -1, 0) + s(q, 0, 0) + s(q, 0, 1)) / 12 * s(vh, 0, 1)
                  + (s(q, -1, 1) + s(q, -1, 0) + s(q, 0, 0)) / 12 * s(vh, -1, 1))
            fv = -(tne * s(uh, 0, 0) + tnw * s(uh, 0, -1) + (s(q, 1, 0) + s(q, 0, 0) + s(q, 0, -1)) / 12 * s(uh, 1, 0)
                   + (s(q, 0, 0) + s(q, 0, -1) + s(q, 1, -1)) / 12 * s(uh, 1, -1))
        else:
            fu = 0.5 * (s(q, 0, 0) + s(q, -1, 0)) * 0.25 * (s(vh, 0, 0) + s(vh, 0, 1) + s(vh, -1, 0) + s(vh, -1, 1))
            fv = -0.5 * (s(q, 0, 0) + s(q, 0, -1)) * 0.25 * (s(uh, 0, 0) + s(uh, 0, -1) + s(uh, 1, 0) + s(uh, 1, -1))
        nu = kw["lateral_viscosity"]
        du[:, 1:-1, 1:-1] = fu - (s(P, 0, 1) - s(P, 0, 0)) / dx + nu * s(_lap(u, dx, dy), 0, 0)
        dv[:, 1:-1, 1:-1] = fv - (s(P, 1, 0) - s(P, 0, 0)) / dy + nu * s(_lap(v, dx, dy), 0, 0)
        du[0] += self.wind
        du[-1] -= kw["bottom_drag"] * u[-1]
        dv[-1] -= kw["bottom_drag"] * v[-1]
        return dh, du, dv


def _masked_exact(case, seed):
    """Conjugate gradients on the masked 5-point operator, to round-off."""
    mask, d, lam = _masked_args(case)
    m = torch.nn.functional.pad(_f64(mask), (1, 1, 1, 1))
    lam = _f64(lam)[:, None, None]
    b = -torch.nn.functional.pad(_f64(_masked_rhs(case, seed)), (1, 1, 1, 1)) * m * d * d

    def op(p):
        out = torch.zeros_like(p)
        c = p[:, 1:-1, 1:-1]
        out[:, 1:-1, 1:-1] = (4.0 * c - p[:, 1:-1, 2:] - p[:, 1:-1, :-2] - p[:, 2:, 1:-1] - p[:, :-2, 1:-1]
                              + lam * d * d * c)
        return out * m

    def dot(a, c):
        return (a * c).sum(dim=(1, 2), keepdim=True)

    x, r = torch.zeros_like(b), b.clone()
    p, rr = r.clone(), dot(b, b)
    target = 1e-28 * rr
    for i in range(8 * (case["nx"] + case["ny"])):
        ap = op(p)
        a = rr / dot(p, ap).clamp_min(1e-300)
        x, r = x + a * p, r - a * ap
        new = dot(r, r)
        p, rr = r + new / rr.clamp_min(1e-300) * p, new
        if i % 32 == 31 and bool((rr <= target).all()):
            break
    return x[:, 1:-1, 1:-1]


def exact(case, seed):
    kind, op = case["kind"], case["op"]
    if kind == "masked":
        return _masked_exact(case, seed).cpu()
    if kind == "ensemble":
        out = []
        for kw, nl, s in _members(case, seed):
            e = _QGExact(case, kw, nl)
            q = _f64(_random_q(case, kw, nl, s).astype(np.float32))
            out.append(_advance(lambda y, e=e: (e.rhs(y[0]),), (q,), case["dt"], case["steps"], case["solver"])[0].cpu())
        return out
    if kind in ("swm", "nonlinear_swm"):
        e = _SWMExact(case)
        y = tuple(_f64(a) for a in _swm_fields(case, seed))
        if op == "rhs":
            y = e.rhs(y)
        else:
            if op == "integrate":
                y = e.boundary(y)
            y = _advance(e.rhs, y, _swm_dt(case), case["steps"], case["solver"])
    else:
        kw = _qg_args(case)
        e = _QGExact(case, kw, case["nl"])
        q = _f64(_random_q(case, kw, case["nl"], seed).astype(np.float32))
        if op == "diagnose":
            y = e.diagnose(q)
            if kind == "barotropic":
                y = tuple(a[0] for a in y)
            return [a.cpu() for a in y]
        if op == "rhs":
            y = (e.rhs(q),)
        else:
            y = _advance(lambda z: (e.rhs(z[0]),), (_inside(q) if op == "integrate" else q,), case["dt"], case["steps"],
                         case["solver"])
    if kind in ("barotropic", "nonlinear_swm"):
        y = tuple(a[0] for a in y)
    if op == "integrate":
        y = tuple(a[None] for a in y)
    return [a.cpu() for a in y]
