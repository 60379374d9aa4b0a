"""GPU tests of which form an inversion takes and of what each form accepts."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from oracle import dst

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


def _member(nx, ny, nl, **kw):
    from somax_amd import testcases as tc

    return tc.ensemble_member(nx, nl, 0.08, ny=ny, **kw)


class _Plan:
    """A QG plan of Nx x Ny points through the C ABI: identity projections, one
    Helmholtz parameter per layer, ghost ring of psi kept."""

    def __init__(self, Nx, Ny, dx, dy, lambdas, precision):
        from somax_amd import _lib
        from somax_amd.qg import _PREC

        self.lib = _lib.load()
        self.nl, self.Ny, self.Nx = len(lambdas), Ny, Nx
        self.f64 = precision == "fp64"
        keep = []

        def dp(a):
            keep.append(np.ascontiguousarray(a, dtype=np.float64))
            return keep[-1].ctypes.data_as(_lib.c_double_p)

        d = _lib.QGDesc()
        d.nx, d.ny, d.nl, d.dx, d.dy = Nx - 2, Ny - 2, self.nl, dx, dy
        d.cl2m, d.cm2l, d.lambdas = dp(np.eye(self.nl)), dp(np.eye(self.nl)), dp(lambdas)
        d.beta_y_row, d.wind_row, d.wind_scale = dp(np.zeros(Ny)), dp(np.zeros(Ny)), dp(np.zeros(self.nl))
        d.advection, d.precision = _lib.ADV_ARAKAWA, _PREC[precision]
        self.plan = ctypes.c_void_p()
        _lib.check(self.lib.somaxhip_qg_plan_create(ctypes.byref(d), ctypes.byref(self.plan)), "plan")
        self.ws_bytes = int(self.lib.somaxhip_qg_workspace_bytes(self.plan))

    def __del__(self):
        self.lib.somaxhip_qg_plan_destroy(self.plan)

    def tensor(self, q):
        import torch

        return torch.from_numpy(q).cuda().to(torch.float64 if self.f64 else torch.float32)

    def invert(self, q, ws_offset=0):
        """psi of the tensor q; the workspace starts ws_offset bytes into an allocation."""
        import torch

        from somax_amd import _lib

        ws = torch.empty(self.ws_bytes + 256, dtype=torch.uint8, device="cuda")
        psi = torch.empty_like(q)
        f = self.lib.somaxhip_qg_invert_f64 if self.f64 else self.lib.somaxhip_qg_invert
        _lib.check(f(self.plan, q.data_ptr(), psi.data_ptr(), 0, ws.data_ptr() + ws_offset, None), "invert")
        torch.cuda.synchronize()
        return psi


@pytest.mark.parametrize("precision", ["fp32", "mixed", "bf16x6", "fp64"])
def test_negative_helmholtz_parameter(gpu, precision):
    """lambda = -2 / dx^2 lies between eigenvalues of the Laplacian on 46 x 46 points,
    0.0042 / dx^2 from the nearest, where the solution is as good as any; -1 / dx^2 twice
    is what an axis' padding modes must not add up to."""
    N, d = 46, 2.0e4
    lams = np.array([-2.0, 0.0]) / d**2
    q = (np.random.default_rng(3).standard_normal((2, N, N)) * 1e-10).astype(np.float32)
    plan = _Plan(N, N, d, d, lams, precision)
    psi = plan.invert(plan.tensor(q)).cpu().numpy()
    for p in range(2):
        r = rel(psi[p], dst.helmholtz_dst(q[p].astype(np.float64), d, d, lams[p]))
        print(f"[forms] lambda {lams[p] * d * d:+.0f} / dx^2, {precision}: rel-L2 {r:.2e}", flush=True)
        assert r < (1e-11 if plan.f64 else 1e-7)
