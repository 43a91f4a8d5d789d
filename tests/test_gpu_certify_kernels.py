"""The certification apply, the projection and C^H at the edges of their launch rules (GPU).

The reference apply against the oracle at 1e-13 of max|K u| (the operator tests' bar) on grids whose planes and
marches end in the middle of a block, and, on larger ones, against the row-march at the same bar; the projection on
both sides of its 256-row rule; C^H of a grid that is no multiple of the kernel's 32 and 256 elements.
"""
import numpy as np
import pytest
import torch

import pgj
from oracle import design, hex8
from pgj import _lib

pytestmark = pytest.mark.gpu
C0 = hex8.isotropic(15 / 26, 5 / 13)


@pytest.mark.parametrize('grid, loads', [((2, 2, 2), 1), ((100, 2, 2), 2), ((3, 17, 16), 1), ((5, 7, 9), 3),
                                         ((19, 20, 21), 2)])
def test_reference_apply_matches_oracle(grid, loads):
    print(f'reference apply {grid}', flush=True)
    rng = np.random.default_rng(sum(grid))
    a = rng.uniform(1e-4, 1, grid)
    voxel = (0.7, 1.1, 0.4)
    op = pgj.Operator(torch.tensor(a, device='cuda'), voxel)
    u = rng.standard_normal((loads, 3 * a.size))
    q = op.apply_reference(torch.tensor(u, device='cuda')).cpu().numpy()
    ref = hex8.apply(a, u, C0, voxel)
    assert np.abs(q - ref).max() < 1e-13 * np.abs(ref).max()


# 4, 8 and 16 planes per march
@pytest.mark.parametrize('grid, loads', [((62, 64, 64), 2), ((61, 64, 64), 4), ((70, 64, 96), 6)])
def test_reference_apply_matches_row_march(grid, loads):
    print(f'reference apply {grid}', flush=True)
    gen = torch.Generator(device='cuda').manual_seed(5)
    a = 1e-4 + torch.rand(grid, generator=gen, device='cuda', dtype=torch.float64)
    op = pgj.Operator(a)
    u = torch.randn((loads, 3 * a.numel()), generator=gen, device='cuda', dtype=torch.float64)
    q, ref = op.apply_reference(u), op.apply_batched(u)
    assert (q - ref).abs().max() < 1e-13 * ref.abs().max()


@pytest.mark.parametrize('grid, loads', [((16, 16, 256), 2), ((41, 41, 39), 2), ((2, 3, 2), 1)])
def test_projection_matches_numpy(grid, loads):
    print(f'projection {grid}', flush=True)
    v = np.random.default_rng(1).standard_normal((loads, 3 * int(np.prod(grid)))) + 3
    op = pgj.Operator(torch.ones(grid, dtype=torch.float64, device='cuda'))
    z = op.project_zero_mean(torch.tensor(v, device='cuda')).cpu().numpy()
    assert np.abs(z - hex8.project(v)).max() < 1e-13 * np.abs(v).max()


@pytest.mark.parametrize('grid', [(2, 3, 5), (5, 6, 9), (8, 8, 8), (9, 10, 12)])
def test_effective_tensor_matches_oracle(grid):
    print(f'effective tensor {grid}', flush=True)
    rng = np.random.default_rng(sum(grid))
    a = rng.uniform(1e-4, 1, grid)
    u = .01 * rng.standard_normal((6, 3 * a.size))
    r = pgj.Resident(grid)
    r.material(torch.tensor(a, device='cuda'))
    r.solutions.copy_(torch.tensor(u))
    H = r.effective_tensor().cpu().numpy()
    ref = design.effective_tensor(a, u, C0)
    assert np.abs(H - ref).max() < 1e-13 * np.abs(ref).max()
