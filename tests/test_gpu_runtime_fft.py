"""The runtime-shaped FFT passes on boxes that use each radix, odd and even x, part chunks and every chunk width (GPU).

The preconditioner is compared with the oracle's to the bar of the other preconditioner tests (1e-13, relative).
"""
import numpy as np
import pytest
import torch

import pgj
from oracle import design, green, hex8

pytestmark = pytest.mark.gpu
C0 = hex8.isotropic(15 / 26, 5 / 13)
# (nz, ny, nx): radices 2..10 alone and together; x odd (no packing) and even; lines that fill a wavefront (128, 256), the
# one length whose group takes two butterflies per lane (243), the largest planes, and cubes between the compile-time ones
BOXES = [(2, 3, 2), (4, 5, 6), (7, 8, 9), (10, 9, 14), (3, 2, 243), (2, 243, 3), (243, 2, 2), (256, 4, 6), (5, 128, 100),
         (27, 25, 49), (45, 60, 50), (75, 14, 63), (6, 81, 98), (20, 20, 20), (40, 40, 40), (100, 12, 80)]


@pytest.mark.parametrize('grid', BOXES, ids=str)
@pytest.mark.parametrize('loads', [1, 7])
def test_runtime_passes_match_oracle(grid, loads):
    print(f'runtime fft {grid} loads={loads}', flush=True)
    rng = np.random.default_rng(sum(grid))
    a = np.exp(rng.uniform(-3, 0, grid))
    G6 = green.symbol(grid, hex8.voxel_of(grid), 15 / 26, 5 / 13)
    r = rng.standard_normal((loads, 3 * a.size))
    pick = sorted({0, loads - 1})
    for alpha in (0.0, 0.5):
        op = pgj.set_alpha(pgj.build(torch.tensor(a, device='cuda')), alpha)
        z = op.apply_precond(torch.tensor(r, device='cuda')).cpu().numpy()[pick]
        ref = green.precond(r[pick], G6, grid, None if alpha == 0 else green.scale(a, alpha, C0))
        assert np.linalg.norm(z - ref) < 1e-13 * np.linalg.norm(ref), (grid, alpha)


@pytest.mark.parametrize('grid', [(9, 10, 7), (20, 14, 30)], ids=str)
def test_runtime_passes_in_the_resident_solve(grid):
    """SoA vectors, the PCG updates and the stop tests: a certified solve whose C^H equals the generic driver's."""
    a = torch.tensor(np.exp(np.random.default_rng(3).uniform(-4, 0, grid)), device='cuda')
    res = pgj.Resident(grid, load_mode='parallel', batch=3).capture()
    res.material(a)
    res.select(0.5)
    infos, _ = res.solve(1e-11)
    assert all(i['converged'] for i in infos)
    op = pgj.set_alpha(pgj.build(a), 0.5)
    for l in (0, 5):
        u, info = pgj.certified_solve(op, op.compute_rhs(np.eye(6)[l]), rtol=1e-11)
        v = res.solutions[l]
        # both residuals are below 1e-11 |f|; the error is at most the condition number of the contrast (e^4) times that
        assert float((u.reshape(-1) - v).norm() / v.norm()) < 1e-8, (grid, l)
        assert abs(info['iterations'] - infos[l]['iterations']) <= 2
