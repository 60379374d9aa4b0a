"""GPU tests of the stripe form of a solve (its first three transforms in one
launch) at the edges of its tiles.

A merged ensemble launches every transform by itself; a single model takes the
stripes where they fit.  Every output's chain of products is the same, so one
step is equal bit for bit.  Six products are held to the 1e-6 of the inversion.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import qg as oqg

pytestmark = pytest.mark.gpu

# N = n + 2 points (half of them, folded, from 256 on): tiles of 32 rows begin and
# end, one or two rows lie past a multiple of 128, k ends in each part of a chunk,
# four and eight tiles are full, and the last fits no more
SHAPES = [(29, 31), (30, 62), (95, 33), (126, 126), (127, 60), (128, 127), (60, 128), (190, 193), (255, 256),
          (254, 254), (256, 254), (254, 256), (256, 400), (450, 322), (510, 256), (512, 512), (514, 512), (516, 514)]


def _member(nx, ny, nl, **kw):
    from somax_amd import testcases as tc

    return tc.ensemble_member(nx, nl, 0.08, ny=ny, **kw)


@pytest.mark.parametrize("nx,ny", SHAPES)
def test_stripes_equal_single_transforms(gpu, nx, ny):
    import torch

    from somax_amd import QGEnsemble
    from somax_amd import testcases as tc

    models = [_member(nx, ny, nl, precision="mixed") for nl in (3, 1)]
    qs = [tc.random_pv(m, 5 + i).astype(np.float32) for i, m in enumerate(models)]
    ens = QGEnsemble(models, merged=True, graph=False)
    packed = ens.pack(qs)
    ens.step(packed, 600.0, 2)
    for i, (m, q) in enumerate(zip(models, qs)):
        one = torch.from_numpy(q).cuda()
        m._step_inplace(one, 600.0, 2)
        assert torch.equal(ens.member(packed, i), one), (nx, ny, i)


@pytest.mark.parametrize("precision", ["bf16x6", "mixed"])
@pytest.mark.parametrize("nx,ny", SHAPES)
def test_stripes_match_oracle(gpu, nx, ny, precision):
    import torch

    from somax_amd import BaroclinicQGState
    from somax_amd import testcases as tc

    model = _member(nx, ny, 2, precision=precision)
    q = tc.random_pv(model, 9).astype(np.float32)
    psi = model.diagnose(BaroclinicQGState(q=torch.from_numpy(q).cuda())).psi.cpu().numpy()
    args = {k: v for k, v in tc.ensemble_member_args(nx, 2, 0.08, ny=ny).items() if k != "n_layers"}
    ref = oqg.invert_pv(oqg.baroclinic_setup(**args), q.astype(np.float64))
    r = float(np.linalg.norm(psi - ref) / np.linalg.norm(ref))
    assert r < 1e-6, (nx, ny, precision, r)


def test_stripes_from_two_streams(gpu):
    """One plan's solves on two streams at once, each with its own workspace."""
    import torch

    from somax_amd import testcases as tc

    model = _member(256, 200, 2, precision="mixed")
    q = torch.from_numpy(tc.random_pv(model, 3).astype(np.float32)).cuda()
    ref = q.clone()
    model._step_inplace(ref, 600.0, 3)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = [q.clone() for _ in streams]
    torch.cuda.synchronize()
    models = [model, _member(256, 200, 2, precision="mixed")]
    for s, o, m in zip(streams, outs, models):
        with torch.cuda.stream(s):
            m._step_inplace(o, 600.0, 3)
    torch.cuda.synchronize()
    assert all(torch.equal(o, ref) for o in outs)
