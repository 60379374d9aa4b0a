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
