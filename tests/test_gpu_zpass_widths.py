"""The forms of the z pass on the compile-time cubes, on either side of the rules that pick them (GPU).

By default the pass runs in registers wherever 16 divides n, except for one FP64 load at 64^3; an explicit radix plan,
the ragged cube 24^3 and that one load take the LDS form (at 64^3 FP64 on the wide chunks from five or six loads on).
The preconditioner of the first and last load is compared with the oracle's, to the bar of the other preconditioner
tests (1e-13 of max|z|); both sides share the loads, so they are also compared with each other.
"""
import numpy as np
import pytest
import torch

import pgj
from oracle import design, green, hex8
from pgj import _lib
from pgj.operator import scale

pytestmark = pytest.mark.gpu
C0 = hex8.isotropic(15 / 26, 5 / 13)


@pytest.fixture
def z_plan():
    """Sets the z pass's FP64 plan on a grid; the default again afterwards."""
    used = []

    def put(grid, plan):
        used.append(grid)
        _lib.check(_lib.lib().pgj_fft_set_plan(grid, 8, 1, plan))
    yield put
    for grid in used:
        _lib.check(_lib.lib().pgj_fft_set_plan(grid, 8, 1, -1))


# (n, loads and plan of one side, loads and plan of the other)
@pytest.mark.parametrize('n, one, other', [(16, (2, -1), (3, 0)), (24, (1, -1), (27, 1)), (32, (5, -1), (5, 1)),
                                           (48, (1, -1), (2, 1)), (64, (1, -1), (2, -1)), (64, (1, 2), (6, 1)),
                                           (96, (1, -1), (1, 1)), (128, (1, -1), (1, 1))])
@pytest.mark.parametrize('scaled', [True, False])
def test_preconditioner_on_both_sides_of_the_z_pass_rules(z_plan, n, one, other, scaled):
    print(f'z pass n={n} loads/plan {one} {other} scaled={scaled}', flush=True)
    grid = (n, n, n)
    a = design.simp(design.filtered_noise(n, 20261104 + n, 2), 1e-4)
    op = pgj.build(torch.tensor(a, device='cuda'))
    s = scale(op, .5) if scaled else None
    most = max(one[0], other[0])
    r = torch.tensor(np.random.default_rng(n).standard_normal((most, 3 * n ** 3)), device='cuda')
    z = []
    for L, plan in (one, other):
        z_plan(op.grid, plan)
        shat = op.scale_spectrum(s) if scaled else None
        z.append(op.green_precond(r[:L].contiguous(), s, shat).cpu().numpy())
    G6 = green.symbol(grid, hex8.voxel_of(grid), 15 / 26, 5 / 13)
    so = green.scale(a, .5, C0) if scaled else None
    for k, L in enumerate((one[0], other[0])):
        pick = sorted({0, L - 1})
        ref = green.precond(r[pick].cpu().numpy(), G6, grid, so)
        err = np.abs(z[k][pick] - ref).max() / np.abs(ref).max()
        assert err < 1e-13, (n, L, err)
    both = min(one[0], other[0])
    assert np.abs(z[0][:both] - z[1][:both]).max() <= 2e-13 * np.abs(z[0]).max()
