"""The device latches of batched PCG steps on both sides of the batch count where they take a launch of their own (GPU)."""
import pytest
import torch

from pgj.pcg import _Workspace

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', [torch.float64, torch.float32])
@pytest.mark.parametrize('B, n', [(1, 3000), (5, 700), (32, 300), (33, 300), (300, 40), (2, 262144), (6, 262144), (3, 1)])
def test_latches(B, n, dtype):
    print(f'pcg latches B={B} n={n} {dtype}', flush=True)
    dev = torch.device('cuda')
    g = torch.Generator(device='cuda').manual_seed(B)
    rnd = lambda: torch.rand((B, n), generator=g, device='cuda', dtype=torch.float64).to(dtype) + 0.5
    w = _Workspace(B, n, dev, dtype)
    rhs, r, best = rnd(), torch.empty((B, n), device='cuda', dtype=dtype), torch.zeros((B, n), device='cuda', dtype=dtype)
    w.start(rhs, None, r)
    assert torch.allclose(w.rhs_norm, rhs.double().norm(dim=1), rtol=1e-6)
    u, p = torch.zeros_like(rhs), rhs.clone()
    w.init(r, r, p)
    # p.Ap = 0 makes every step length 0, so the step measures the residuals as they are: tolerance 2e-3, near 2e-2
    # (size of the first residuals, of the last one, states after, which improve)
    steps = [(.1, .1, [0, 0], [True] * B), (1e-3, .2, [0, 0], [True] * (B - 1) + [False]),
             (1e-4, .01, [0, 1], [True] * B), (5e-5, 1e-3, [4, 1], [True] * B), (1e-6, 1e-6, [4, 1], [False] * B)]
    for it, (size, last, state, improves) in enumerate(steps, 1):
        r.copy_(rhs * size)
        r[-1] = rhs[-1] * last
        u.fill_(float(it))
        before = best.clone()
        w.pre_step(u, r, p, torch.zeros_like(p), best, 2e-3, 2e-2, it, True)
        want = r.double().norm(dim=1) / rhs.double().norm(dim=1)
        assert torch.allclose(w.res, want, rtol=1e-6)
        assert w.state.tolist() == state and w.improved.bool().tolist() == improves
        moved = torch.tensor(improves, device='cuda')
        assert bool((best[moved] == it).all()) and torch.equal(best[~moved], before[~moved])
