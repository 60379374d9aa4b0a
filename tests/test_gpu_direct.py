"""GPU tests of the direct FP64 inversion (somax_amd/csrc/direct.hip).

Its sums and intermediates are FP64, so the FP32 streamfunction it stores is
off by the rounding of the last store alone: at most 2**-24 = 6e-8 of each
value, hence of the 2-norm; the bar of 1e-7 leaves the rest to the FP64 sums.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import qg as oqg

pytestmark = pytest.mark.gpu

BAR = 1e-7

# (nx, ny, nl): folded extents (n + 3) // 2 around the tile of 16 and the
# k-batches of 16 (16, 17, 15, 33), odd and even lines, thin grids, every layer
# instance of the kernels, and the largest extent (304) along either axis
SIZES = [(2, 2, 1), (3, 5, 2), (29, 30, 3), (30, 31, 1), (31, 32, 4), (28, 63, 5), (64, 33, 8), (127, 30, 2),
         (130, 129, 3), (606, 9, 3), (9, 605, 2), (254, 256, 3)]


@pytest.mark.parametrize("mass", [False, True])
@pytest.mark.parametrize("nx,ny,nl", SIZES)
def test_direct_inversion_matches_oracle(gpu, nx, ny, nl, mass):
    import torch

    from somax_amd import BaroclinicQG

    H = tuple(float(h) for h in np.linspace(300.0, 700.0, nl))
    gp = (9.81,) + tuple(0.03 / (1.0 + k) for k in range(nl - 1))
    kw = dict(nx=nx, ny=ny, Lx=2e4 * nx, Ly=3e4 * ny, H=H, g_prime=gp)
    model = BaroclinicQG.create(n_layers=nl, mass_correction=mass, **kw)
    setup = oqg.baroclinic_setup(mass_correction=mass, **kw)
    q = (np.random.default_rng(nx * 1000 + ny).standard_normal((nl, ny + 2, nx + 2)) * 1e-6).astype(np.float32)
    for bc in (False, True):
        psi = model._invert(torch.from_numpy(q).cuda(), bc).cpu().numpy().astype(np.float64)
        q64 = oqg.apply_bc(q) if bc else q.astype(np.float64)
        ref = oqg.invert_pv(setup, q64)
        r = float(np.linalg.norm(psi - ref) / np.linalg.norm(ref))
        print(f"[direct] {nx}x{ny}x{nl} mass={mass} bc={bc}: psi {r:.2e}", flush=True)
        assert r < BAR


# around the limits of the one-launch front (rows and row at most 64, 8192 points
# over the layers): on it 126 x 126 x 2, 127 x 125, 64 x 64 x 8 and 30 x 78 x 2 (one
# tile of columns, three of rows); past it 129 x 126, 126 x 129, 126 x 126 x 3
FRONT = [(126, 126, 1), (127, 125, 1), (129, 126, 1), (126, 129, 1), (64, 64, 5), (64, 64, 6), (64, 64, 8), (30, 78, 2), (126, 126, 2),
         (126, 126, 3)]


@pytest.mark.parametrize("nx,ny,nl", FRONT)
def test_direct_front_equals_the_two_launches(gpu, nx, ny, nl):
    """The front kernel takes the same sums in the same order as the forward and
    spectral kernels, and serves at most 256 workgroups: the members of an
    ensemble large enough for the two launches equal the single model's step bit
    for bit, and its inversion meets the oracle (bar as above)."""
    import torch

    from somax_amd import BaroclinicQG, QGEnsemble

    H = tuple(float(h) for h in np.linspace(300.0, 700.0, nl))
    gp = (9.81,) + tuple(0.03 / (1.0 + k) for k in range(nl - 1))
    kw = dict(nx=nx, ny=ny, Lx=2e4 * nx, Ly=3e4 * ny, H=H, g_prime=gp)
    members = 256 // (nl * 4 * ((nx + 3) // 2 + 15 >> 4)) + 1
    models = [BaroclinicQG.create(n_layers=nl, **kw) for _ in range(members)]
    rng = np.random.default_rng(nx * 1000 + ny)
    qs = [(rng.standard_normal((nl, ny + 2, nx + 2)) * 1e-6).astype(np.float32) for _ in range(members)]
    setup = oqg.baroclinic_setup(**kw)
    for bc in (False, True):
        psi = models[0]._invert(torch.from_numpy(qs[0]).cuda(), bc).cpu().numpy().astype(np.float64)
        ref = oqg.invert_pv(setup, oqg.apply_bc(qs[0]) if bc else qs[0].astype(np.float64))
        r = float(np.linalg.norm(psi - ref) / np.linalg.norm(ref))
        print(f"[direct] front {nx}x{ny}x{nl} bc={bc}: psi {r:.2e}", flush=True)
        assert r < BAR
    ens = QGEnsemble(models, graph=False)
    packed = ens.pack(qs)
    ens.step(packed, 600.0, 1)
    for i in (0, members // 2, members - 1):
        q = torch.from_numpy(qs[i]).cuda()
        models[i]._step_inplace(q, 600.0, 1)
        assert torch.equal(ens.member(packed, i), q.view(ens.shapes[i])), i
