"""GPU tests of the 64 x 64 transform tiles (launches of few tiles).

A single model's launches take them; the classes of a concurrent ensemble keep
the 128-wide tiles.  Every output's chain of products is the same, so a mixed
member equals its single model bit for bit.  The FP32 tiles are held to the
1e-6 that the FP32 inversion meets elsewhere.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import qg as oqg

pytestmark = pytest.mark.gpu

# N = n + 2 (or its half, folded) around multiples of 32, 64 and 128, where the
# tiles, the k-tiles and the fringe of one or two rows begin and end
SIZES = [(29, 31), (62, 63), (64, 126), (127, 128), (130, 190), (253, 65), (254, 256), (258, 382), (400, 130)]


def _member(nx, ny, nl, **kw):
    from somax_amd import testcases as tc

    return tc.ensemble_member(nx, nl, 0.08, ny=ny, **kw)


@pytest.mark.parametrize("nx,ny", SIZES)
def test_small_tiles_equal_wide_tiles(gpu, nx, ny):
    import torch

    from somax_amd import QGEnsemble
    from somax_amd import testcases as tc

    models = [_member(nx, ny, 3, precision="mixed"), _member(40, 36, 1, precision="mixed")]
    qs = [tc.random_pv(m, 5 + i).astype(np.float32) for i, m in enumerate(models)]
    ens = QGEnsemble(models, concurrent=True, graph=False)
    assert ens.num_classes == 2
    packed = ens.pack(qs)
    ens.step(packed, 600.0, 1)
    for i, (m, q) in enumerate(zip(models, qs)):
        one = torch.from_numpy(q).cuda()
        m._step_inplace(one, 600.0, 1)
        assert torch.equal(ens.member(packed, i), one), (nx, ny, i)


@pytest.mark.parametrize("precision", ["fp32", "bf16x6"])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_small_tiles_match_oracle(gpu, nx, ny, precision):
    import torch

    from somax_amd import BaroclinicQGState
    from somax_amd import testcases as tc

    model = _member(nx, ny, 2, precision=precision)
    q = tc.random_pv(model, 9).astype(np.float32)
    psi = model.diagnose(BaroclinicQGState(q=torch.from_numpy(q).cuda())).psi.cpu().numpy()
    args = {k: v for k, v in tc.ensemble_member_args(nx, 2, 0.08, ny=ny).items() if k != "n_layers"}
    ref = oqg.invert_pv(oqg.baroclinic_setup(**args), q.astype(np.float64))
    r = float(np.linalg.norm(psi - ref) / np.linalg.norm(ref))
    print(f"[small tiles] {nx}x{ny} {precision}: psi {r:.2e}", flush=True)
    assert r < 1e-6
