"""The z pass's kx chunk widths on either side of the rule that picks them (GPU).

The compile-time cubes run narrow chunks while the default ones give at most 2.5 blocks per CU, the default
chunks above that (at 64^3 FP64 the wide ones from 6 loads on). The preconditioner of the first and last load is
compared with the oracle's, to the bar of the other preconditioner tests (1e-13 of max|z|); both sides of the rule
share the loads, so they are also compared with each other.
"""
import numpy as np
import pytest
import torch

import pgj
from oracle import design, green, hex8
from pgj.operator import scale

pytestmark = pytest.mark.gpu
C0 = hex8.isotropic(15 / 26, 5 / 13)


# at 256 CUs the rule changes between these load counts (640 default blocks)
@pytest.mark.parametrize('n, below, above', [(16, 40, 41), (24, 26, 27), (32, 20, 21), (48, 1, 6), (64, 3, 4),
                                             (64, 1, 6)])
@pytest.mark.parametrize('scaled', [True, False])
def test_preconditioner_on_both_sides_of_the_width_rule(n, below, above, scaled):
    print(f'z widths n={n} loads {below}/{above} scaled={scaled}', flush=True)
    grid = (n, n, n)
    a = design.simp(design.filtered_noise(n, 20261104 + n, 2), 1e-4)
    op = pgj.build(torch.tensor(a, device='cuda'))
    s = scale(op, .5) if scaled else None
    shat = op.scale_spectrum(s) if scaled else None
    r = torch.tensor(np.random.default_rng(n).standard_normal((above, 3 * n ** 3)), device='cuda')
    z = [op.green_precond(r[:L].contiguous(), s, shat).cpu().numpy() for L in (below, above)]
    G6 = green.symbol(grid, hex8.voxel_of(grid), 15 / 26, 5 / 13)
    so = green.scale(a, .5, C0) if scaled else None
    for k, L in enumerate((below, above)):
        pick = sorted({0, L - 1})
        ref = green.precond(r[pick].cpu().numpy(), G6, grid, so)
        err = np.abs(z[k][pick] - ref).max() / np.abs(ref).max()
        assert err < 1e-13, (n, L, err)
    assert np.abs(z[0] - z[1][:below]).max() <= 2e-13 * np.abs(z[0]).max()
