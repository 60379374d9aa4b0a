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


@pytest.mark.parametrize("precision", ["fp32", "mixed", "bf16x6", "fp64"])
@pytest.mark.parametrize("Nx,Ny", [(5, 4), (23, 50), (46, 33), (66, 67), (131, 67), (257, 40), (130, 130), (260, 262),
                                   (303, 218), (514, 258)])
def test_workspace_contents_do_not_matter(gpu, Nx, Ny, precision):
    """An inversion and a right-hand side from a workspace of NaN equal those from one of
    zeros, bit for bit: no form reads what it has not written."""
    import torch

    from somax_amd import _lib

    lams = np.array([0.0, 3e-10])
    plan = _Plan(Nx, Ny, 2e4, 3e4, lams, precision)
    q = plan.tensor((np.random.default_rng(Nx + Ny).standard_normal((2, Ny, Nx)) * 1e-10).astype(np.float32))
    prm = _lib.QGParams(15.0, 1e9, 3.6e-8, 0.0)
    rhs = plan.lib.somaxhip_qg_rhs_f64 if plan.f64 else plan.lib.somaxhip_qg_rhs
    outs = []
    for byte in (0, 255):
        ws = torch.full((plan.ws_bytes,), byte, dtype=torch.uint8, device="cuda")
        psi, psi2, dq = (torch.empty_like(q) for _ in range(3))
        inv = plan.lib.somaxhip_qg_invert_f64 if plan.f64 else plan.lib.somaxhip_qg_invert
        for bc in (1, 0):
            ws.fill_(byte)
            _lib.check(inv(plan.plan, q.data_ptr(), psi.data_ptr(), bc, ws.data_ptr(), None), "invert")
            ws.fill_(byte)
            _lib.check(rhs(plan.plan, q.data_ptr(), dq.data_ptr(), psi2.data_ptr(), ctypes.byref(prm), bc,
                           ws.data_ptr(), None), "rhs")
            outs.append([psi.clone(), psi2.clone(), dq.clone()])
    for a, b in zip(outs[:2], outs[2:]):
        assert all(torch.isfinite(x).all() and torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("Nx,Ny", [(34, 40), (131, 67), (258, 258), (303, 218), (514, 100)])
def test_workspace_aligned_to_eight_bytes(gpu, Nx, Ny, precision):
    """A workspace that starts 8 bytes past an allocation's start gives the bits of an
    aligned one, in inversions and right-hand sides."""
    import torch

    from somax_amd import _lib

    plan = _Plan(Nx, Ny, 2e4, 3e4, np.array([0.0, 3e-10]), precision)
    q = plan.tensor((np.random.default_rng(Nx + Ny).standard_normal((2, Ny, Nx)) * 1e-10).astype(np.float32))
    rhs = plan.lib.somaxhip_qg_rhs_f64 if plan.f64 else plan.lib.somaxhip_qg_rhs
    prm = _lib.QGParams(15.0, 1e9, 3.6e-8, 0.0)
    outs = []
    for offset in (0, 8):
        ws = torch.empty(plan.ws_bytes + 256, dtype=torch.uint8, device="cuda")
        dq = torch.empty_like(q)
        _lib.check(rhs(plan.plan, q.data_ptr(), dq.data_ptr(), None, ctypes.byref(prm), 1, ws.data_ptr() + offset,
                       None), "rhs")
        torch.cuda.synchronize()
        outs.append((plan.invert(q, offset), dq))
    assert all(torch.equal(x, y) for x, y in zip(*outs))


# (precision, n, layers, members): grids whose steps invert in the direct form (256^2 FP32,
# 64^2 and 144^2 six products, 511^2) and by the transforms (512^2, 192^2), with members
# enough that the class leaves the launch shapes of a single model
SIBLINGS = [("fp32", 256, 3, 33), ("fp32", 512, 3, 3), ("fp32", 511, 2, 5), ("fp32", 430, 1, 8), ("bf16x6", 64, 3, 30),
            ("bf16x6", 144, 2, 14), ("bf16x6", 192, 3, 4), ("mixed", 200, 3, 5)]


@pytest.mark.parametrize("merged", [False, True])
@pytest.mark.parametrize("precision,n,nl,members", SIBLINGS)
def test_member_bits_do_not_depend_on_siblings(gpu, precision, n, nl, members, merged):
    """A member steps as its single model does, bit for bit, in a class of many planes
    and beside a class of another grid."""
    import torch

    from somax_amd import QGEnsemble
    from somax_amd import testcases as tc

    models = [_member(n, n, nl, precision=precision)] * members + [_member(48, 40, 2, precision=precision)]
    pv = [tc.random_pv(m, 7 + i).astype(np.float32) for i, m in enumerate((models[0], models[-1]))]
    qs = [pv[0] * np.float32(1.0 + 0.01 * i) for i in range(members)] + [pv[1]]
    ens = QGEnsemble(models, merged=merged)
    packed = ens.pack(qs)
    ens.step(packed, 600.0, 2)
    for i in (0, members // 2, members - 1, members):
        one = torch.from_numpy(qs[i]).cuda()
        models[i]._step_inplace(one, 600.0, 2)
        assert torch.equal(ens.member(packed, i), one.view(ens.shapes[i])), i
