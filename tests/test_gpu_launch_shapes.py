"""GPU tests of launch shapes that the choice rules keep apart elsewhere: the same
outputs, bit for bit, from another tile height, tile size, grouping or stream, and
the FP64 instances of the direct inversion at its extents."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from oracle import qg as oqg

pytestmark = pytest.mark.gpu


def _member(nx, ny, nl, **kw):
    from somax_amd import testcases as tc

    return tc.ensemble_member(nx, nl, 0.08, ny=ny, **kw)


def _fields(models):
    from somax_amd import testcases as tc

    return [tc.random_pv(m, 5 + i).astype(np.float32) for i, m in enumerate(models)]


def _same_as_single(models, nsteps=1, **kw):
    import torch

    from somax_amd import QGEnsemble

    qs = _fields(models)
    ens = QGEnsemble(models, graph=False, **kw)
    packed = ens.pack(qs)
    ens.step(packed, 600.0, nsteps)
    for i, (m, q) in enumerate(zip(models, qs)):
        one = torch.from_numpy(q).cuda()
        m._step_inplace(one, 600.0, nsteps)
        assert torch.equal(ens.member(packed, i), one.view(ens.shapes[i])), i


# a merged group's stage kernel keeps 16 rows; a single model takes 4, 8 or 16
@pytest.mark.parametrize("nx,ny", [(63, 4), (64, 5), (65, 16), (66, 17), (126, 31), (256, 336), (256, 352), (448, 768),
                                   (448, 784)])
def test_weno_heights_equal_the_merged_group(gpu, nx, ny):
    kw = dict(precision="mixed", advection="weno")
    _same_as_single([_member(nx, ny, 3, **kw), _member(40, 36, 1, **kw)], merged=True)


# grids whose mixed solves take single launches, past the stripes' extents (258 points
# plain, 516 folded); around multiples of 32, 64 and 128 and with a fringe of one or
# two rows.  A single model's few tiles are 64 x 64, a concurrent class' 128 wide.
@pytest.mark.parametrize("nx,ny", [(259, 30), (261, 62), (301, 131), (318, 255), (383, 127), (403, 259), (518, 516),
                                   (522, 524), (574, 700), (640, 514)])
def test_small_tiles_of_single_launches_equal_wide_tiles(gpu, nx, ny):
    _same_as_single([_member(nx, ny, 2, precision="mixed"), _member(40, 36, 1, precision="mixed")])


# merged groups of the direct form: more than eight column tiles (two a workgroup), six
# products, and classes that fall into a direct and a transform group
GROUPS = {
    "wide": ("fp32", [(300, 64, 3), (256, 256, 2), (511, 130, 1), (20, 40, 3)]),
    "deep": ("fp32", [(256, 64, 5), (290, 30, 1), (64, 64, 8)]),
    "six": ("bf16x6", [(64, 64, 3), (96, 40, 2), (144, 144, 1), (20, 300, 2)]),
    "split": ("fp32", [(512, 512, 1), (256, 256, 3), (448, 430, 2), (64, 600, 2)]),
    "six split": ("bf16x6", [(256, 256, 3), (64, 64, 2), (200, 160, 1)]),
}


@pytest.mark.parametrize("case", sorted(GROUPS))
def test_merged_direct_groups_equal_single_models(gpu, case):
    precision, shapes = GROUPS[case]
    kw = dict(precision=precision)
    if case == "deep":
        from somax_amd import BaroclinicQG

        models = []
        for nx, ny, nl in shapes:
            H = tuple(float(h) for h in np.linspace(300.0, 700.0, nl))
            gp = (9.81,) + tuple(0.03 / (1.0 + k) for k in range(nl - 1))
            models.append(BaroclinicQG.create(nx=nx, ny=ny, n_layers=nl, Lx=2e4 * nx, Ly=2e4 * ny, H=H, g_prime=gp,
                                              mass_correction=True, **kw))
    else:
        models = [_member(nx, ny, nl, **kw) for nx, ny, nl in shapes]
    _same_as_single(models, nsteps=2, merged=True)


@pytest.mark.parametrize("precision", ["fp32", "mixed", "bf16x6"])
def test_one_plan_on_two_streams(gpu, precision):
    """Steps and inversions of one plan on two streams at once, a workspace each: the
    operators and tables are all that they share."""
    import torch

    from somax_amd import _lib

    model = _member(256, 200, 2, precision=precision)
    q = torch.from_numpy(_fields([model])[0]).cuda()
    ref = q.clone()
    model._step_inplace(ref, 600.0, 3)
    psi_ref = model._invert(ref, True).clone()
    torch.cuda.synchronize()
    lib, plan, prm = _lib.load(), model._ensure_plan(), model._c_params()
    nbytes = int(lib.somaxhip_qg_workspace_bytes(plan))
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = [(q.clone(), torch.empty_like(q), torch.empty(nbytes, dtype=torch.uint8, device="cuda")) for _ in streams]
    torch.cuda.synchronize()
    for s, (o, psi, ws) in zip(streams, outs):
        st = ctypes.c_void_p(s.cuda_stream)
        _lib.check(lib.somaxhip_qg_step(plan, o.data_ptr(), None, 3, 600.0, ctypes.byref(prm), ws.data_ptr(), st), "step")
        _lib.check(lib.somaxhip_qg_invert(plan, o.data_ptr(), psi.data_ptr(), 1, ws.data_ptr(), st), "invert")
    torch.cuda.synchronize()
    for o, psi, _ in outs:
        assert torch.equal(o, ref) and torch.equal(psi, psi_ref)


# as the FP32 sizes of the direct form; the bar: sums of up to 608 terms in four
# products, 2**-53 each (2.7e-13 if none cancelled), with room for the mode mix
@pytest.mark.parametrize("mass", [False, True])
@pytest.mark.parametrize("nx,ny,nl", [(2, 2, 1), (3, 5, 2), (29, 30, 3), (30, 31, 1), (31, 32, 4), (28, 63, 5), (64, 33, 8),
                                      (127, 30, 2), (130, 129, 3), (606, 9, 3), (9, 605, 2), (254, 256, 3), (604, 606, 1)])
def test_direct_fp64_inversion_matches_oracle(gpu, nx, ny, nl, mass):
    import torch

    from somax_amd import BaroclinicQG

    H = tuple(float(h) for h in np.linspace(300.0, 700.0, nl))
    gp = (9.81,) + tuple(0.03 / (1.0 + k) for k in range(nl - 1))
    kw = dict(nx=nx, ny=ny, Lx=2e4 * nx, Ly=3e4 * ny, H=H, g_prime=gp)
    model = BaroclinicQG.create(n_layers=nl, mass_correction=mass, precision="fp64", **kw)
    setup = oqg.baroclinic_setup(mass_correction=mass, **kw)
    q = np.random.default_rng(nx * 1000 + ny).standard_normal((nl, ny + 2, nx + 2)) * 1e-6
    for bc in (False, True):
        psi = model._invert(torch.from_numpy(q).cuda(), bc).cpu().numpy()
        ref = oqg.invert_pv(setup, oqg.apply_bc(q) if bc else q)
        r = float(np.linalg.norm(psi - ref) / np.linalg.norm(ref))
        print(f"[direct] fp64 {nx}x{ny}x{nl} mass={mass} bc={bc}: psi {r:.2e}", flush=True)
        assert r < 1e-12
