"""GPU tests of the stage kernels at the edges of their tiles.

A tile is 64 columns by 4, 8 or 16 rows of the interior block (4 rows for the
shallow-water stage); the ghost ring is stored by the edge tiles or by
workgroups of its own.  A single model chooses the height by its number of
tiles, the classes of an ensemble keep 16 rows, and every height gives the same
bits.  One step is held to the 1e-6 relative L2 that the steps meet elsewhere.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import qg as oqg
from oracle import swm as oswm

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


def _member(nx, ny, nl, **kw):
    from somax_amd import testcases as tc

    return tc.ensemble_member(nx, nl, 0.08, ny=ny, **kw)


# remainders of 64 columns and of 4, 8 and 16 rows; the last four lie on both
# sides of the two lines of the rule (256 and 1024 tiles of 16 rows, 3 layers)
SHAPES = [(63, 4), (64, 5), (65, 16), (66, 17), (126, 31), (256, 336), (256, 352), (448, 768), (448, 784)]


@pytest.mark.parametrize("advection", ["arakawa", "weno"])
@pytest.mark.parametrize("nx,ny", SHAPES)
def test_stage_heights_give_the_same_bits(gpu, nx, ny, advection):
    import torch

    from somax_amd import QGEnsemble
    from somax_amd import testcases as tc

    kw = dict(precision="mixed", advection=advection)
    models = [_member(nx, ny, 3, **kw), _member(40, 36, 1, **kw)]
    qs = [tc.random_pv(m, 5 + i).astype(np.float32) for i, m in enumerate(models)]
    ens = QGEnsemble(models, concurrent=True, graph=False)
    packed = ens.pack(qs)
    ens.step(packed, 600.0, 1)
    one = torch.from_numpy(qs[0]).cuda()
    models[0]._step_inplace(one, 600.0, 1)
    assert torch.equal(ens.member(packed, 0), one)


@pytest.mark.parametrize("precision,advection", [("fp32", "arakawa"), ("fp32", "weno"), ("mixed", "weno"),
                                                 ("fp64", "arakawa")])
@pytest.mark.parametrize("nx,ny", [(63, 4), (65, 17), (256, 352), (448, 784)])
def test_tsit5_ragged_grid_matches_oracle(gpu, nx, ny, precision, advection):
    import torch

    from somax_amd import testcases as tc

    model = _member(nx, ny, 2, precision=precision, advection=advection)
    args = {k: v for k, v in tc.ensemble_member_args(nx, 2, 0.08, ny=ny).items() if k != "n_layers"}
    setup = oqg.baroclinic_setup(advection=advection, **args)
    q = tc.random_pv(model, 9).astype(np.float32)
    qd = torch.from_numpy(q).cuda().to(torch.float64 if precision == "fp64" else torch.float32)
    model._step_tsit5_inplace(qd, 600.0, 2)
    ref = q.astype(np.float64)
    for _ in range(2):
        ref = oqg.tsit5_step(setup, ref, 600.0)
    assert rel(qd.cpu().numpy(), ref) < (1e-12 if precision == "fp64" else 2e-6)


@pytest.mark.parametrize("solver", ["ssprk3", "tsit5"])
@pytest.mark.parametrize("nx,ny,bc,flux", [(61, 3, "wall", "energy_enstrophy"), (62, 4, "periodic", "energy_enstrophy"),
                                           (64, 5, "channel", "average"), (65, 66, "periodic", "average"),
                                           (126, 9, "channel", "energy_enstrophy"), (129, 8, "wall", "average"),
                                           (200, 130, "periodic", "energy_enstrophy")])
def test_swm_ragged_grid_steps_match_oracle(gpu, nx, ny, bc, flux, solver):
    """Three layers, one call of 1 step and one of 3 (which carries the
    thickness deviation between its steps)."""
    import torch

    from somax_amd import MultilayerShallowWater2D, MultilayerSW2DState

    args = dict(nx=nx, ny=ny, Lx=1e4 * nx, Ly=1e4 * ny, f0=1e-4, beta=1e-11, H=(400.0, 1100.0, 2500.0),
                g_prime=(9.81, 0.025, 0.0125), bc=bc, lateral_viscosity=20.0, bottom_drag=1e-7,
                wind_amplitude=2e-5, vorticity_flux=flux)
    model = MultilayerShallowWater2D.create(n_layers=3, **args)
    s = oswm.setup(**args)
    rng = np.random.default_rng(nx * 10 + ny)
    h = (np.asarray(s.H)[:, None, None] + rng.standard_normal(s.shape)).astype(np.float32)
    u = (0.2 * rng.standard_normal(s.shape)).astype(np.float32)
    v = (0.2 * rng.standard_normal(s.shape)).astype(np.float32)
    dt = 0.3 * 1e4 / np.sqrt(9.81 * 4000.0)
    step = oswm.ssprk3_step if solver == "ssprk3" else oswm.tsit5_step
    for n in (1, 3):
        out = model.step(MultilayerSW2DState(*(torch.from_numpy(a.copy()).cuda() for a in (h, u, v))), dt, n,
                         solver=solver)
        ref = [a.astype(np.float64) for a in (h, u, v)]
        for _ in range(n):
            ref = step(s, *ref, dt)
        assert max(rel(a.cpu().numpy(), b) for a, b in zip((out.h, out.u, out.v), ref)) < n * 1e-6
