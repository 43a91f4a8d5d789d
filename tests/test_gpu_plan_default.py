"""Plan 0 is the library's own choice of each FFT pass, so that queried plans can be set back (GPU)."""
import numpy as np
import pytest
import torch

import pgj
from pgj import _lib, tune

pytestmark = pytest.mark.gpu


def _set(grid, es, plans):
    for pas, plan in enumerate(plans):
        _lib.check(_lib.lib().pgj_fft_set_plan(grid, es, pas, plan))


# 16: radix 4 first and the z pass in registers; 24: the LDS z pass; 64: either by the load count
@pytest.mark.parametrize('n, batch', [(16, 2), (24, 2), (32, 2), (64, 1), (64, 2)])
def test_queried_plans_set_back_change_nothing(n, batch):
    print(f'plans set back {n}^3 batch {batch}', flush=True)
    r = pgj.Resident(n, loads=np.eye(6)[:batch], load_mode='parallel')
    a = torch.tensor(np.exp(np.random.default_rng(n).uniform(-4, 0, (n, n, n))), device='cuda')
    out = []
    try:
        for back in (False, True):
            plans = tune.fft_plans(r.op.grid, 8)
            assert plans == (0, 0, 0)
            if back:
                _set(r.op.grid, 8, plans)
            r.material(a)
            r.select('0.5')
            r._setup(range(batch), 1e-300)
            r.u.zero_()
            r.certify()
            r.initialize()
            r.iteration(4)
            out.append(r.u.clone())
    finally:
        _set(r.op.grid, 8, (-1, -1, -1))
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize('plans', [(3, 3, 3), (1, 1, 1), (3, 1, 0)])
@pytest.mark.parametrize('n', [16, 48, 64])
def test_explicit_schedules_agree(n, plans):
    """Radix 4 first (3) and radix 8 first (1): the iterates of the default to rounding."""
    print(f'schedules {plans} {n}^3', flush=True)
    r = pgj.Resident(n, loads=np.eye(6)[:2], load_mode='parallel')
    r.material(torch.tensor(np.exp(np.random.default_rng(n).uniform(-4, 0, (n, n, n))), device='cuda'))
    r.select('0.5')
    out = []
    try:
        for p in ((0, 0, 0), plans):
            _set(r.op.grid, 8, p)
            assert tune.fft_plans(r.op.grid, 8) == p
            r._setup(range(2), 1e-300)
            r.u.zero_()
            r.certify()
            r.initialize()
            r.iteration(4)
            out.append(r.u.clone())
    finally:
        _set(r.op.grid, 8, (-1, -1, -1))
    assert float((out[0] - out[1]).abs().max()) < 1e-10 * float(out[0].abs().max())
