"""The FP64 row march with two x per lane on cubic voxels: shapes of four, two and one row waves, long and short marches,
part rounds; the apply against the independent thread-per-node kernel, p.Kp against its own sums (GPU)."""
import numpy as np
import pytest
import torch

import pgj
from pgj import _lib

pytestmark = pytest.mark.gpu


def _shape(op, L):
    import ctypes
    out = (ctypes.c_int * 5)()
    _lib.check(_lib.lib().pgj_hex8_get_shape(op.grid, L, 8, out))
    return tuple(out)


# (grid, loads, row waves, planes per block) the rule picks
@pytest.mark.parametrize('grid, loads, W, ZC', [((5, 7, 66), 1, 1, 1), ((9, 6, 70), 2, 2, 1), ((64, 64, 128), 1, 2, 4),
                                                ((128, 128, 128), 1, 4, 16), ((96, 96, 96), 3, 4, 32)], ids=str)
def test_apply_matches_the_reference_kernel(grid, loads, W, ZC):
    print(f'pair march {grid} loads={loads}', flush=True)
    rng = np.random.default_rng(sum(grid))
    a = torch.tensor(np.exp(rng.uniform(-6, 0, grid)), device='cuda')
    op = pgj.Operator(a, (0.01,) * 3)
    R, w, z, plane, _ = _shape(op, loads)
    assert (R, w, z, plane) == (1, W, ZC, 1)
    u = torch.tensor(rng.standard_normal((loads, 3 * a.numel())), device='cuda')
    got, ref = op.apply_batched(u), op.apply_reference(u)
    # each force is a sum of 8 x 24 terms no larger than the largest: 192 roundings of 1.1e-16 in the worst case
    assert float((got - ref).abs().max()) < 192 * 1.2e-16 * float(ref.abs().max()) * 2


def test_quadratic_form_in_the_native_steps():
    """p.Kp is summed from values read again at the store: a wrong one would change the step lengths at once."""
    a = torch.tensor(np.exp(np.random.default_rng(7).uniform(-3, 0, (8, 8, 96))), device='cuda')
    op = pgj.set_alpha(pgj.Operator(a, (0.02,) * 3).enable_green(), 0.5)
    rhs = op.compute_rhs(np.eye(6)[4])

    class Plain:
        apply, apply_precond = staticmethod(op.apply), staticmethod(op.apply_precond)
    u, it, _ = pgj.solve_pcg_batched(op, rhs, tol=1e-30, max_iter=9)
    v, jt, _ = pgj.solve_pcg_batched(Plain, rhs, tol=1e-30, max_iter=9)
    assert it == jt == 9 and float((u - v).norm() / v.norm()) < 1e-9
