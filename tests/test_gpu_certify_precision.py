"""The certification apply is no less accurate than the operator it certifies (GPU).

Rounding errors of both against the stiffness and the sums in extended precision, on displacements whose rigid part
is large beside their strains (a smooth field over many voxels, with and without an offset), where forms that cancel
the rigid part in rounded coefficients lose digits.
"""
import numpy as np
import pytest
import torch

import pgj

pytestmark = pytest.mark.gpu
LAM, MU = 15 / 26, 5 / 13


def _stiffness(h):
    """24x24 Ke in extended precision: products of the axes' mass, stiffness and mixed integrals."""
    h = np.asarray(h, np.longdouble)
    mass = [[x / 3, x / 6] for x in h]
    K = np.zeros((24, 24), np.longdouble)
    sign = lambda n, i: 1 if (n >> i) & 1 else -1
    for n in range(8):
        for m in range(8):
            d = [(n ^ m) >> i & 1 for i in range(3)]
            D = np.zeros((3, 3), np.longdouble)   # integral of dN_n/dx_i dN_m/dx_j
            for i in range(3):
                for j in range(3):
                    if i == j:
                        D[i, i] = np.longdouble(sign(n, i) * sign(m, i)) / h[i]
                        for k in range(3):
                            if k != i:
                                D[i, i] *= mass[k][d[k]]
                    else:
                        D[i, j] = np.longdouble(sign(n, i) * sign(m, j)) / 4 * mass[3 - i - j][d[3 - i - j]]
            block = LAM * D + MU * D.T + MU * np.trace(D) * np.eye(3, dtype=np.longdouble)
            K[3 * n:3 * n + 3, 3 * m:3 * m + 3] = block
    return K


def _exact(a, u, h):
    K = _stiffness(h)
    grid = a.shape
    f = u.reshape(*grid, 3).astype(np.longdouble)
    corner = [(-(n >> 2), -(n >> 1 & 1), -(n & 1)) for n in range(8)]
    local = [np.roll(f, s, (0, 1, 2)) for s in corner]
    out = np.zeros_like(f)
    for n in range(8):
        force = sum(local[m] @ K[3 * n:3 * n + 3, 3 * m:3 * m + 3].T for m in range(8)) * a[..., None]
        out += np.roll(force, tuple(-s for s in corner[n]), (0, 1, 2))
    return out.reshape(-1)


@pytest.mark.parametrize('grid, voxel', [((32, 32, 32), None), ((20, 24, 40), (.7, 1.1, .4)), ((9, 5, 64), None)])
@pytest.mark.parametrize('offset', [0., 3.])
def test_reference_apply_is_as_accurate_as_the_row_march(grid, voxel, offset):
    print(f'certification apply {grid} offset {offset}', flush=True)
    rng = np.random.default_rng(2)
    a = 1e-4 + rng.random(grid)
    z, y, x = (2 * np.pi * c / c.size for c in np.ogrid[:grid[0], :grid[1], :grid[2]])
    z, y, x = np.broadcast_arrays(z, y, x)
    u = np.stack([.05 * np.sin(x + d) * np.cos(y - d) + .03 * np.sin(2 * z + d) for d in range(3)], axis=-1)
    u = (u + .1 / max(grid) * (rng.random(u.shape) - .5) + offset).reshape(1, -1)
    op = pgj.Operator(torch.tensor(a, device='cuda'), voxel)
    ud = torch.tensor(u, device='cuda')
    ref = _exact(a, u[0], (op.mesh.dx, op.mesh.dy, op.mesh.dz))
    err = [float(np.linalg.norm((q.cpu().numpy()[0] - ref).astype(float)) / np.linalg.norm(ref.astype(float)))
           for q in (op.apply_reference(ud), op.apply_batched(ud))]
    print(f'  relative error: certification {err[0]:.2e}, row march {err[1]:.2e}', flush=True)
    assert err[0] <= err[1]
