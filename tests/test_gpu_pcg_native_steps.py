"""Iterations of ``solve_pcg_batched`` run by one library call against the same loop over the operator's methods (GPU).

The two differ in how p.Ap and r.z are summed, so iterates agree to rounding amplified by the solve; both are checked
against the same tolerance on the residual.
"""
import numpy as np
import pytest
import torch

import pgj

pytestmark = pytest.mark.gpu


class _Plain:
    """The operator's methods without its class, so that the loop calls them one by one."""

    def __init__(self, op):
        self.op, self.mesh = op, op.mesh
        self.calls = 0

    def apply(self, u):
        self.calls += 1
        return self.op.apply(u)

    def apply_precond(self, r):
        return self.op.apply_precond(r)


def _problem(grid, alpha, seed=1):
    a = torch.tensor(np.exp(np.random.default_rng(seed).uniform(-4, 0, grid)), device='cuda')
    op = pgj.set_alpha(pgj.build(a), alpha)
    return op, op.compute_rhs(np.eye(6)[3])


# compile-time cubes, runtime boxes (odd x, x of two per lane), an x for which the apply has no row march (75)
@pytest.mark.parametrize('grid', [(16, 16, 16), (24, 24, 24), (5, 7, 9), (12, 10, 14), (4, 6, 96), (6, 4, 75)], ids=str)
@pytest.mark.parametrize('alpha', [0.0, 0.5])
@pytest.mark.parametrize('options', [dict(), dict(update_mode='compiled', convergence_check_stride=4),
                                     dict(update_mode='compiled', convergence_check_stride=5,
                                          convergence_check_adaptive_factor=10.0)], ids=['eager', 'stride 4', 'adaptive'])
def test_native_steps_equal_the_loop(grid, alpha, options):
    print(f'native steps {grid} alpha={alpha} {options}', flush=True)
    op, rhs = _problem(grid, alpha)
    plain = _Plain(op)
    u, it, res = pgj.solve_pcg_batched(op, rhs, tol=1e-9, max_iter=900, **options)
    v, jt, ser = pgj.solve_pcg_batched(plain, rhs, tol=1e-9, max_iter=900, **options)
    assert plain.calls >= jt and abs(it - jt) <= 1
    assert float(res.max()) < 1e-9 and float(ser.max()) < 1e-9
    # two iterates within 1e-9 of the right-hand side: apart by at most 2e-9 times the condition number, about e^4
    assert float((u - v).norm() / v.norm()) < 1e-6
    u, it, _ = pgj.solve_pcg_batched(op, rhs, tol=1e-30, max_iter=7, x0=v, **options)
    w, jt, _ = pgj.solve_pcg_batched(plain, rhs, tol=1e-30, max_iter=7, x0=v, **options)
    assert it == jt == 7 and float((u - w).norm() / w.norm()) < 1e-8


def test_replaced_methods_are_called():
    op, rhs = _problem((8, 8, 8), 0.5)
    ref, it, _ = pgj.solve_pcg_batched(op, rhs, tol=1e-8)
    calls = []
    apply, precond = op.apply, op.apply_precond
    op.apply_precond = lambda r: (calls.append('m'), precond(r))[1]
    u, jt, _ = pgj.solve_pcg_batched(op, rhs, tol=1e-8)
    assert len(calls) == jt and jt == it
    op.apply_precond = precond
    op.apply = lambda p: (calls.append('k'), apply(p))[1]
    u, jt, _ = pgj.solve_pcg_batched(op, rhs, tol=1e-8)
    assert calls.count('k') == jt == it and float((u - ref).norm() / ref.norm()) < 1e-6
