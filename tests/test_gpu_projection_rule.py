"""The zero-mean projection on both sides of the rule that reduces the means in a launch of their own (GPU): more than
1400 blocks in all and more than 256 partial rows per load. Same bar as the other projection tests."""
import numpy as np
import pytest
import torch

import pgj
from oracle import hex8

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('grid, loads', [((41, 41, 39), 5), ((41, 41, 39), 6), ((64, 64, 64), 1), ((70, 72, 72), 1),
                                         ((40, 40, 40), 6)])
def test_projection_matches_numpy(grid, loads):
    print(f'projection {grid} {loads}', flush=True)
    v = np.random.default_rng(1).standard_normal((loads, 3 * int(np.prod(grid)))) + 3
    op = pgj.Operator(torch.ones(grid, dtype=torch.float64, device='cuda'))
    z = op.project_zero_mean(torch.tensor(v, device='cuda')).cpu().numpy()
    assert np.abs(z - hex8.project(v)).max() < 1e-13 * np.abs(v).max()
